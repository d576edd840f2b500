"""Batched on-GPU speech-to-text (Whisper) - replaces the reference's external
OpenAI-compatible STT round trip (``stt_client.go:207-362``: float32->WAV encode,
multipart POST, JSON decode) with: pinned PCM16 -> H2D -> fused convert+RMS
kernel -> log-mel -> encoder -> greedy decoder, batched across utterances.

Random-init weights cannot produce a real transcript, so benchmark/synthetic
requests carry their known transcript and the decoder is *teacher-forced* to it:
every step still runs the full decoder forward and the
argmax over the 51 866-entry vocabulary, so cost is that of a real greedy decode
of the same length; only the fed-back token is the reference one.
"""
from __future__ import annotations

import logging
import os
import queue
import threading
import time
from concurrent.futures import FIRST_COMPLETED, Future, ThreadPoolExecutor, wait
from dataclasses import dataclass, field

import numpy as np
import torch

from .. import ops
from ..models.configs import WhisperConfig
from ..models.whisper import WhisperModel, WhisperWeights, decode_step_fast, decode_step_fused
from ..utils.tracing import tracer
from .batching import join_futures, plan_step
from .kv_cache import PagedKVCache
from .tokenizer import get_tokenizer

log = logging.getLogger("loqa.stt")

N_SAMPLES = 480000  # 30 s @ 16 kHz
# numpy PCM of direct submissions staged through the pinned stager (False: a
# one-off pinned tensor copy per request)
PCM_STAGER = True
# relay PCM copied to HBM chunk by chunk while the relay speaks (pcm_staging.py)
PCM_STREAM_IN = os.environ.get("LOQA_PCM_STREAM_IN", "1") != "0"
# long-form audio: an utterance longer than 30 s is split into
# 30 s windows, encoded as extra encoder rows of the same batch (one
# cross-attention slot each) and decoded window after window, each window's
# decode prompted with the previous window's text (<|startofprev|>, at most
# PREV_TOKENS tokens, fed 4 per step like the SOT prompt); the texts are joined.
MAX_WINDOWS = int(os.environ.get("LOQA_STT_MAX_WINDOWS", "20"))
PREV_TOKENS = int(os.environ.get("LOQA_STT_PREV_TOKENS", "32"))
# admissions that may pass a waiting item that does not fit yet (FIFO otherwise)
HOL_BYPASS = int(os.environ.get("LOQA_STT_HOL_BYPASS", "16"))


def n_windows(n_samples: int, cap: int = MAX_WINDOWS) -> int:
    """30 s windows of an utterance, at most ``cap`` (an engine passes
    min(MAX_WINDOWS, max_batch): every window holds a cross-attention slot, so
    a longer utterance is truncated like one past MAX_WINDOWS, not rejected)."""
    return max(1, min(cap, -(-n_samples // N_SAMPLES)))


@dataclass(eq=False)
class STTRequest:
    pcm: np.ndarray                   # int16 samples @ 16 kHz
    transcript: str | None = None     # teacher-forcing target (synthetic mode)
    max_new_tokens: int = 96          # per 30 s window
    staged: object = None             # pinned PCM slot (engine/pcm_staging.py) holding the samples
    n_samples: int = 0                # samples uploaded (<= MAX_WINDOWS x 30 s)
    # teacher-forcing targets per 30 s window of a long-form utterance (else
    # ``transcript`` is split over the windows by words)
    transcript_windows: list | None = None
    # outputs
    text: str = ""
    sumsq: float = 0.0
    rms: float = 0.0
    tokens: list[int] = field(default_factory=list)
    seq_id: int = -1
    t_done: float = 0.0
    t_enc0: float = 0.0               # encoder start / end, decoder start (perf_counter)
    t_enc1: float = 0.0
    t_dec0: float = 0.0
    # decoder state (engine-owned)
    slot: int = -1                    # cross-attention K|V slot (encoder rows)
    target: list[int] | None = None
    feed: list[int] = field(default_factory=list)
    step: int = 0
    on_done: object = None
    # long-form state (engine-owned): windows, the one being decoded, their
    # cross-attention slots, finished windows' texts / tokens, prompt steps
    windows: int = 1
    win: int = 0
    slots: list = field(default_factory=list)
    win_texts: list = field(default_factory=list)
    prev_tokens: list = field(default_factory=list)
    prompt_steps: int = 1


class STTEngine:
    SEQ_BUCKETS = [1, 2, 4, 8, 16, 32, 64, 128]
    SPLIT_KEYS = 128
    RES_SLOTS = 3       # result ring slots (>= steps in flight + 1)

    def __init__(self, cfg: WhisperConfig, device, *, seed: int = 0, max_batch: int = 64,
                 block_size: int = 16, use_graphs: bool = True, fast_decode: bool = True,
                 fused: bool = True, weights: WhisperWeights | None = None,
                 contended_tuning: bool = False, tokenizer=None, language: str = "en"):
        self.cfg = cfg
        self.device = torch.device(device)
        if self.device.type == "cuda" and self.device.index is None:
            self.device = torch.device("cuda", torch.cuda.current_device())
        from ..utils.streams import decode_cap, init_pools
        init_pools(self.device)       # fixed stream -> hardware-queue placement
        self.max_wgs = decode_cap("LOQA_STT_MAX_WGS")
        # optional: tune the decode GEMMs under a background weight stream
        # (ops.contended_tuning; measured noisier and 5 % slower end to end)
        with ops.decode_cap(self.max_wgs), ops.contended_tuning(self.device, contended_tuning):
            self.weights = weights or WhisperWeights(cfg, self.device, seed=seed)
        self.weights.max_wgs = self.max_wgs or ops.MAX_DECODE_WGS
        self.model = WhisperModel(self.weights)
        self.tok = tokenizer or get_tokenizer(cfg.vocab_size)
        # start-of-transcript prompt; the language token follows STT_LANGUAGE
        # (the reference passes it to its STT service)
        try:
            lang = self.tok.token_id(f"<|{language}|>")
        except KeyError:
            raise ValueError(f"STT language {language!r}: no <|{language}|> token in the "
                             "tokenizer (a multilingual Whisper tokenizer.json has one)") from None
        self.sot = [self.tok.token_id("<|startoftranscript|>"), lang,
                    self.tok.token_id("<|transcribe|>"), self.tok.token_id("<|notimestamps|>")]
        self.eot = self.tok.token_id("<|endoftext|>")
        self.n_prompt_tokens_per_step = len(self.sot)
        try:
            self.sop = self.tok.token_id("<|startofprev|>")
        except KeyError:
            self.sop = None     # no previous-text prompt for long-form windows
        # a checkpoint's tokenizer: greedy decoding never emits its special /
        # timestamp tokens or the generation config's suppress_tokens (as the
        # reference's STT service decodes); one packed mask row for every
        # sequence. The synthetic tokenizer of the random-init weights: none.
        self._sup = self._sup_rows = None
        if hasattr(self.tok, "sampling_mask"):
            from ..ops.reference import pack_mask
            self._sup = pack_mask(self.tok.sampling_mask(keep=(self.eot,))[None]).to(self.device)
            self._sup_rows = torch.zeros(max(256, 2 * max_batch), dtype=torch.int32,
                                         device=self.device)
        self.block_size = block_size
        self.max_blocks = (cfg.n_text_ctx + block_size - 1) // block_size
        self.kv = PagedKVCache(cfg.dec_layers, cfg.n_heads, cfg.head_dim,
                               max_batch * self.max_blocks + 8, block_size, self.device)
        self.is_gpu = self.device.type == "cuda"
        self.ws = ops.AttnWorkspace(self.device, max_batch * 8, cfg.n_heads, cfg.head_dim,
                                    max((cfg.n_audio_ctx + 255) // 256, (cfg.n_text_ctx + 255) // 256)
                                    ) if self.is_gpu else None
        self._next = 1
        self.stats = {"utterances": 0, "decode_steps": 0, "host_pre_s": 0.0, "gpu_wait_s": 0.0,
                      "encode_s": 0.0}
        self.max_batch = max_batch
        self.fast_decode = fast_decode
        # fused-epilogue decoder GEMMs (8 launches per layer) for Mpad <= 64
        self.fused = fused and fast_decode
        self.scratch = ops.FusedScratch(self.device) if self.fused else None
        self.use_graphs = use_graphs and self.is_gpu and fast_decode
        self.self_splits = (cfg.n_text_ctx + self.SPLIT_KEYS - 1) // self.SPLIT_KEYS
        # cross-attention keys per split (the workspace holds n_audio_ctx / 128 splits)
        self.cross_split_keys = max(self.SPLIT_KEYS,
                                    int(os.environ.get("LOQA_XATTN_SPLIT_KEYS", "256")) // 32 * 32)
        if fast_decode and self.is_gpu:
            self.ws = ops.AttnWorkspace(self.device, 128, cfg.n_heads, cfg.head_dim,
                                        max(self.self_splits, (cfg.n_audio_ctx + self.SPLIT_KEYS - 1)
                                            // self.SPLIT_KEYS))
        # cross-attention K|V of every decoder layer for up to max_batch
        # utterances, written in place each batch (graph-captured steps read it)
        # (with the layer-concatenated weights: one [rows, L * 2d] buffer whose
        # column blocks are the layers' K|V, written by one tiled GEMM per batch)
        self.xkv_all = None
        if getattr(self.weights, "xkv_all", None) is not None:
            self.xkv_all = torch.empty(max_batch * cfg.n_audio_ctx, cfg.dec_layers * 2 * cfg.d_model,
                                       dtype=torch.bfloat16, device=self.device)
            d2 = 2 * cfg.d_model
            self.xkv = [self.xkv_all[:, i * d2:(i + 1) * d2] for i in range(cfg.dec_layers)]
        else:
            self.xkv = [torch.empty(max_batch * cfg.n_audio_ctx, 2 * cfg.d_model, dtype=torch.bfloat16,
                                    device=self.device) for _ in range(cfg.dec_layers)]
        self._graphs: dict[tuple[int, int], dict] = {}
        self._graphs_frozen = False     # see LLMEngine: no capture while serving
        self._enc_graphs: dict = {}
        self._enc_graph_pool = None
        # token budget of one decoder step (each new sequence feeds the 4-token
        # SOT prompt; 17+ simultaneous arrivals would exceed ops.MPADS rows)
        self.step_tokens = max(len(self.sot), min(int(os.environ.get("LOQA_STT_STEP_TOKENS", "64")),
                                                  ops.MPADS[-2]))
        self._rr = 0
        if self.use_graphs:
            # step I/O without copy-engine operations between step graphs (as the
            # LLM engine: elementwise.hip step_fetch / step_publish): a 2-slot
            # pinned staging ring for the step metadata, a result ring, a device
            # counter of launched step graphs, and the last token of every
            # cross-attention slot (+ a trash slot) for device-fed greedy steps
            b_max = next((b for b in self.SEQ_BUCKETS if b >= max_batch), self.SEQ_BUCKETS[-1])
            self._n32_max = 4 * ops.MPADS[-1] + 6 * b_max + 1 + b_max * self.max_blocks
            self._n64_max = max(16, ops.mpad_for(min(b_max, ops.MPADS[-1])))
            self._stage32 = torch.zeros(2, self._n32_max, dtype=torch.int32).pin_memory()
            self._stage64 = torch.zeros(2, self._n64_max, dtype=torch.int64).pin_memory()
            self._res_ring = torch.zeros(self.RES_SLOTS, 256, dtype=torch.int32).pin_memory()
            self._step_ctr = torch.zeros(1, dtype=torch.int32, device=self.device)
            self._step_no = 0
            self.last_tok = torch.zeros(max_batch + 1, dtype=torch.int32, device=self.device)
        # two decoder steps in flight (the host prepares step j+1 while step j
        # runs); LOQA_STT_PIPELINE=0: one synchronous step at a time
        self.pipelined = self.use_graphs and os.environ.get("LOQA_STT_PIPELINE", "1") != "0"

    # ------------------------------------------------------------ front end
    def upload(self, reqs: list[STTRequest], device_pcm: torch.Tensor | None = None
               ) -> tuple[torch.Tensor, torch.Tensor]:
        """PCM16 of all utterances -> device -> fused convert + pad + sum of
        squares kernel -> [B, 480000] f32 (the 30 s window).

        GPU: every request's samples sit in a pinned stager slot (the relay's
        chunks were appended there as they arrived; numpy requests are staged
        here), each slot goes to HBM with one hipMemcpyAsync on the stager's
        H2D stream, and this (compute) stream waits on the copies' events.
        ``device_pcm`` (already on the GPU, e.g. scattered by the DP router
        over RCCL) holds the concatenated samples and skips the copies."""
        lens = []
        for r in reqs:
            n = self._n_samples(r)
            w = n_windows(n, self.max_windows)
            if n > w * N_SAMPLES:
                self.stats["long_form_dropped_samples"] = \
                    self.stats.get("long_form_dropped_samples", 0) + n - w * N_SAMPLES
                log.error("utterance of %.1f s exceeds %d windows (LOQA_STT_MAX_WINDOWS, "
                          "max_batch): the last %.1f s are not transcribed", n / 16000,
                          self.max_windows, (n - w * N_SAMPLES) / 16000)
            lens.append(min(n, w * N_SAMPLES))
            r.windows = w
        for r, n in zip(reqs, lens):
            r.n_samples = n
        offs = np.zeros(len(reqs) + 1, np.int64)
        offs[1:] = np.cumsum(lens)
        # one padded 30 s encoder row per window: a request's windows are
        # consecutive slices of its samples, so the rows' offsets are the
        # cumulative row lengths
        row_lens = [min(N_SAMPLES, n - w * N_SAMPLES) for r, n in zip(reqs, lens)
                    for w in range(r.windows)]
        row_offs = np.zeros(len(row_lens) + 1, np.int64)
        row_offs[1:] = np.cumsum(row_lens)
        if device_pcm is not None:
            pcm = device_pcm[: int(offs[-1])]
        elif self.is_gpu:
            pcm = torch.empty(max(1, int(offs[-1])), dtype=torch.int16, device=self.device)
            cur = torch.cuda.current_stream(self.device).cuda_stream
            stager = self._stager()
            for r, o, n in zip(reqs, offs[:-1], lens):
                slot = r.staged if r.staged is not None else (
                    stager.stage(r.pcm) if PCM_STAGER else None)
                if slot is None:        # every pinned slot busy: a one-off pinned copy
                    h = torch.from_numpy(np.ascontiguousarray(r.pcm[:n], np.int16)).pin_memory()
                    pcm[int(o):int(o) + n].copy_(h, non_blocking=True)
                    continue
                slot.upload(pcm.data_ptr() + int(o) * 2, n, cur)
                r.staged = None
        else:
            pcm = torch.from_numpy(np.concatenate(
                [np.asarray(self._host_samples(r)[:n], np.int16) for r, n in zip(reqs, lens)]
                or [np.zeros(0, np.int16)]))
            for r in reqs:
                if r.staged is not None:
                    r.staged.release()
                    r.staged = None
        off_t = torch.from_numpy(row_offs)
        if self.is_gpu:
            off_t = off_t.pin_memory().to(self.device, non_blocking=True)
        return ops.pcm16_to_f32_padded(pcm, off_t, N_SAMPLES, row_offs)

    @staticmethod
    def _n_samples(r: STTRequest) -> int:
        return len(r.staged) if r.staged is not None else len(r.pcm)

    @staticmethod
    def _host_samples(r: STTRequest) -> np.ndarray:
        return r.staged.numpy() if r.staged is not None else r.pcm

    def _stager(self):
        """The engine's pinned PCM stager (created on first use)."""
        if getattr(self, "stager", None) is None:
            from .pcm_staging import PcmStager
            h2d = None
            if PCM_STREAM_IN:
                from ..utils.streams import placed_stream
                h2d = placed_stream(self.device, "h2d")
            self.stager = PcmStager(2 * self.max_batch + 16, N_SAMPLES, h2d_stream=h2d)
        return self.stager

    def new_pcm_slot(self):
        """A pinned slot for one relay's incoming PCM (None: CPU engine or every
        slot busy - the caller then buffers on the host)."""
        if not self.is_gpu:
            return None
        return self._stager().acquire()

    # -------------------------------------------------------------- decode
    def cross_kv(self, enc: torch.Tensor, slots: list[int] | None = None) -> list[torch.Tensor]:
        """Cross-attention K|V of every decoder layer for the encoder rows of
        ``enc`` ([n * T_enc, d]), written to the requests' slots (default:
        slots 0..n-1, one GEMM per layer; contiguous slot runs share a GEMM)."""
        T = self.cfg.n_audio_ctx
        n = enc.shape[0] // T
        slots = list(range(n)) if slots is None else slots
        assert max(slots) < self.max_batch, "slot exceeds max_batch"
        runs, i = [], 0                     # (first request, first slot, length)
        while i < n:
            j = i
            while j + 1 < n and slots[j + 1] == slots[j] + 1:
                j += 1
            runs.append((i, slots[i], j - i + 1))
            i = j + 1
        if self.xkv_all is not None:
            w = self.weights
            for i0, s0, m in runs:
                ops.gemm_tile(enc[i0 * T:(i0 + m) * T], w.xkv_all, bias=w.xkv_all_b,
                              out=self.xkv_all[s0 * T:(s0 + m) * T], layout=7)
            return self.xkv
        for L, buf in zip(self.weights.dec, self.xkv):
            for i0, s0, m in runs:
                torch.addmm(L["xkv_b"], enc[i0 * T:(i0 + m) * T], L["xkv"].t(),
                            out=buf[s0 * T:(s0 + m) * T])
        return self.xkv

    def _host_meta(self, live: list[STTRequest], B_pad: int, T_pad: int,
                   out: dict | None = None) -> tuple[int, dict]:
        T_enc = self.cfg.n_audio_ctx
        L = max(16, ops.mpad_for(B_pad))
        if out is not None:  # preallocated pinned views (graph path), filled below
            tokens, positions, slots = out["tokens"], out["positions"], out["slots"]
            cu, ctx, bt = out["cu_q"], out["ctx_lens"], out["block_tables"]
            enc_starts, enc_lens, lidx = out["enc_starts"], out["enc_lens"], out["logit_idx"]
        else:
            tokens = np.zeros(T_pad, np.int32)
            positions = np.zeros(T_pad, np.int32)
            slots = np.full(T_pad, -1, np.int32)
            cu = np.zeros(B_pad + 1, np.int32)
            ctx = np.zeros(B_pad, np.int32)
            bt = np.zeros((B_pad, self.max_blocks), np.int32)
            enc_starts = np.zeros(B_pad, np.int32)
            enc_lens = np.zeros(B_pad, np.int32)
            lidx = np.zeros(L, np.int64)
        T = sum(len(r.feed) for r in live)
        tokens.fill(0)
        if T:
            tokens[:T] = [t for r in live for t in r.feed]
        rc = self.kv.pool.step_meta([r.seq_id for r in live], [len(r.feed) for r in live], B_pad,
                                    T_pad, self.max_blocks, positions, slots, cu, ctx, bt, lidx)
        if rc == -2:
            raise RuntimeError("STT KV cache exhausted")
        if rc != 0:
            raise RuntimeError(f"step metadata failed ({rc})")
        n = len(live)
        enc_starts[:n] = [r.slot * T_enc for r in live]
        enc_starts[n:] = 0
        enc_lens[:n] = T_enc
        enc_lens[n:] = 0
        max_q = max([len(r.feed) for r in live] + [1])
        return max_q, {"tokens": tokens, "positions": positions, "slots": slots, "cu_q": cu,
                       "ctx_lens": ctx, "block_tables": bt, "enc_starts": enc_starts,
                       "enc_lens": enc_lens, "logit_idx": lidx}

    def _dev(self, host: dict, dst: dict | None = None) -> dict:
        out = {}
        for k, a in host.items():
            t = torch.from_numpy(a)
            if self.is_gpu:
                t = t.pin_memory()
            if dst is not None:
                dst[k].copy_(t, non_blocking=True)
                out[k] = dst[k]
            else:
                out[k] = t.to(self.device, non_blocking=True)
        return out

    def _self_splits(self, ctx: int | None) -> int:
        """Self-attention key splits for a context bound (graph bucket)."""
        if ctx is None:
            return self.self_splits
        return max(1, min(self.self_splits, (ctx + self.SPLIT_KEYS - 1) // self.SPLIT_KEYS))

    def _argmax(self, logits: torch.Tensor) -> torch.Tensor:
        if self._sup is None:
            return ops.masked_argmax(logits)
        return ops.masked_argmax(logits, self._sup, self._sup_rows[: logits.shape[0]])

    def _fast_forward(self, dev: dict, max_q: int, B_pad: int, ctx: int | None = None) -> torch.Tensor:
        ns = self._self_splits(ctx)
        if self.fused and dev["tokens"].numel() <= 64:
            logits = decode_step_fused(self.model, dev["tokens"], dev["positions"], dev["slots"],
                                       dev["cu_q"], dev["ctx_lens"], dev["block_tables"], max_q,
                                       self.kv.k, self.kv.v, self.xkv, dev["enc_starts"],
                                       dev["enc_lens"], dev["logit_idx"], self.ws, self.scratch,
                                       ns, self.SPLIT_KEYS, self.cross_split_keys)
            return self._argmax(logits[:B_pad, : self.cfg.vocab_size])
        logits = decode_step_fast(self.model, dev["tokens"], dev["positions"], dev["slots"],
                                  dev["cu_q"], dev["ctx_lens"], dev["block_tables"], max_q,
                                  self.kv.k, self.kv.v, self.xkv, dev["enc_starts"],
                                  dev["enc_lens"], dev["logit_idx"], self.ws, ns,
                                  self.SPLIT_KEYS)
        return self._argmax(logits[:B_pad, : self.cfg.vocab_size])

    def _graph(self, B_pad: int, T_pad: int, ctx: int) -> dict:
        """Captured decode step for (sequence bucket, token bucket, context
        bucket): the attention grid is sized for the bucket's context, so no
        workgroups are spent on splits past the longest sequence. The graph's
        first node fills the step metadata from the pinned staging ring (taking
        a greedy sequence's fed token from ``last_tok`` on the device), its last
        node publishes the sampled tokens to the pinned result ring."""
        key = (B_pad, T_pad, ctx)
        g = self._graphs.get(key)
        if g is not None:
            return g
        shapes = {"tokens": (T_pad,), "positions": (T_pad,), "slots": (T_pad,),
                  "cu_q": (B_pad + 1,), "ctx_lens": (B_pad,),
                  "block_tables": (B_pad, self.max_blocks), "enc_starts": (B_pad,),
                  "enc_lens": (B_pad,), "src": (T_pad,), "row_slot": (B_pad,)}
        n32 = sum(int(np.prod(v)) for v in shapes.values())
        L = max(16, ops.mpad_for(B_pad))
        assert n32 <= self._n32_max and L <= self._n64_max and B_pad <= 256
        d32 = torch.zeros(n32, dtype=torch.int32, device=self.device)
        d64 = torch.zeros(L, dtype=torch.int64, device=self.device)
        dev, off = {}, 0
        for k, shp in shapes.items():
            n = int(np.prod(shp))
            dev[k] = d32[off:off + n].view(*shp)
            off += n
        dev["slots"].fill_(-1)
        dev["src"].fill_(-1)
        dev["row_slot"].fill_(self.max_batch)
        dev["logit_idx"] = d64
        max_q = max(1, min(len(self.sot), T_pad))
        s = torch.cuda.Stream(self.device)
        s.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(s):
            self._fast_forward(dev, max_q, B_pad, ctx)
        torch.cuda.current_stream(self.device).wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        k = ops._lib.kernels()
        lib = ops._lib
        # thread-local capture: the other GPU worker thread keeps running
        with ops.graph_capture(graph, capture_error_mode="thread_local"):
            st = lib.stream_ptr(d32)
            src_off = dev["src"].data_ptr() // 4 - d32.data_ptr() // 4
            lib.check(k.loqa_step_fetch(
                lib.ptr(d32), self._stage32.data_ptr(), n32, self._n32_max, lib.ptr(d64),
                self._stage64.data_ptr(), L, self._n64_max, lib.ptr(self._step_ctr), T_pad, src_off,
                lib.ptr(self.last_tok), st), "step_fetch")
            out = self._fast_forward(dev, max_q, B_pad, ctx)
            lib.check(k.loqa_step_publish(
                lib.ptr(out), B_pad, self._res_ring.data_ptr(), self._res_ring.shape[1],
                self.RES_SLOTS, lib.ptr(self._step_ctr), lib.ptr(dev["row_slot"]),
                lib.ptr(self.last_tok), st), "step_publish")
        g = {"graph": graph, "dev": dev, "out": out, "shapes": shapes, "n32": n32, "L": L}
        self._graphs[key] = g
        return g

    def _stage(self, g: dict) -> dict:
        """Numpy views of the staging slot of the NEXT step-graph launch."""
        slot = self._step_no % 2
        hn, out, off = self._stage32[slot].numpy(), {}, 0
        for k, shp in g["shapes"].items():
            n = int(np.prod(shp))
            out[k] = hn[off:off + n].reshape(shp)
            off += n
        out["logit_idx"] = self._stage64[slot].numpy()[: g["L"]]
        return out

    def _replay(self, g: dict) -> int:
        """Launch a step graph whose staging slot is filled; returns the result
        ring slot its tokens land in."""
        rslot = self._step_no % self.RES_SLOTS
        g["graph"].replay()
        self._step_no = (self._step_no + 1) % (2 * self.RES_SLOTS)   # wraps as the device counter
        return rslot

    # encoder graphs for batches of up to this many utterances (0: eager encoder)
    ENC_GRAPH_MAX = 4

    def _enc_graph(self, B: int) -> dict:
        """The Whisper encoder (log-mel -> conv stem -> all layers) for a batch
        of B padded 30-s windows as ONE graph replay: ~330 kernels per encode
        launched eagerly from the encoder worker thread leave host-launch gaps
        between them (and hold the GIL the decoder schedulers need). The graphs
        share one memory pool; replays run on the encoder's stream one after
        another, so their intermediates never overlap in time."""
        g = self._enc_graphs.get(B)
        if g is not None:
            return g
        if self._enc_graph_pool is None:
            self._enc_graph_pool = torch.cuda.graph_pool_handle()
        audio = torch.zeros(B, 480000, dtype=torch.float32, device=self.device)
        s = torch.cuda.Stream(self.device)
        s.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(s):
            self.model.encode(audio)
        torch.cuda.current_stream(self.device).wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with ops.graph_capture(graph, pool=self._enc_graph_pool, capture_error_mode="thread_local"):
            out = self.model.encode(audio)
        g = {"graph": graph, "audio": audio, "out": out}
        self._enc_graphs[B] = g
        return g

    def encode(self, audio: torch.Tensor) -> torch.Tensor:
        """Encoder states [B * 1500, d] of padded audio [B, 480000]: a graph
        replay for a captured batch size, else the eager encoder."""
        B = audio.shape[0]
        g = self._enc_graphs.get(B)
        if g is None:
            return self.model.encode(audio)
        g["audio"].copy_(audio)
        g["graph"].replay()
        return g["out"]

    def warmup_graphs(self) -> int:
        """Capture every decoder-step graph bucket up front (see
        ``LLMEngine.warmup_graphs``): sequence x token x context buckets; and
        the encoder for batches of 1 .. ``ENC_GRAPH_MAX`` utterances."""
        if not self.use_graphs:
            return 0
        n = 0
        if self.is_gpu:
            for b in range(1, min(self.ENC_GRAPH_MAX, self.max_batch) + 1):
                self._enc_graph(b)
                n += 1
        n_sot = len(self.sot)
        b_max = next((b for b in self.SEQ_BUCKETS if b >= self.max_batch), self.SEQ_BUCKETS[-1])
        for b in self.SEQ_BUCKETS:
            if b > b_max:
                break
            t_min = ops.mpad_for(min(self.step_tokens, b // 2 + 1))   # T >= B > b/2
            t_max = ops.mpad_for(min(self.step_tokens, b * n_sot))
            for t in ops.MPADS:
                if t > t_max:
                    break
                if t < t_min:
                    continue
                for c in range(self.SPLIT_KEYS, self.cfg.n_text_ctx + self.SPLIT_KEYS, self.SPLIT_KEYS):
                    self._graph(b, t, min(c, self.cfg.n_text_ctx))
                    n += 1
        self._graphs_frozen = True
        return n

    def _step(self, live: list[STTRequest]) -> np.ndarray:
        """One decoder step for every live request (its ``feed`` tokens)."""
        B = len(live)
        T = sum(len(r.feed) for r in live)
        if self.fast_decode:
            B_pad = next((b for b in self.SEQ_BUCKETS if b >= B), B)
            T_pad = ops.mpad_for(T)
            ctx = max(self.kv.pool.seq_len(r.seq_id) + len(r.feed) for r in live)
            C = min(self.cfg.n_text_ctx, -(-ctx // self.SPLIT_KEYS) * self.SPLIT_KEYS)
            if self.use_graphs and ((B_pad, T_pad, C) in self._graphs or not self._graphs_frozen):
                t0 = time.perf_counter()
                g = self._graph(B_pad, T_pad, C)
                hb = self._stage(g)
                self._host_meta(live, B_pad, T_pad, out=hb)
                hb["src"].fill(-1)
                hb["row_slot"].fill(self.max_batch)
                t1 = time.perf_counter()
                rslot = self._replay(g)
                torch.cuda.current_stream(self.device).synchronize()
                out = self._res_ring[rslot, :B].numpy().copy()
                self.stats["host_pre_s"] += t1 - t0
                self.stats["gpu_wait_s"] += time.perf_counter() - t1
                return out
            max_q, host = self._host_meta(live, B_pad, T_pad)
            return self._fast_forward(self._dev(host), max_q, B_pad)[:B].cpu().numpy()
        return self._eager_step(live)

    def _eager_step(self, live: list[STTRequest]) -> np.ndarray:
        """Reference decode path (hipBLASLt GEMMs, eager launches)."""
        T_enc = self.cfg.n_audio_ctx
        toks, pos, slots, cu, ctx, lidx = [], [], [], [0], [], []
        bt = np.zeros((len(live), self.max_blocks), np.int32)
        max_q, max_ctx = 1, 1
        for j, r in enumerate(live):
            f = r.feed
            start = self.kv.pool.seq_len(r.seq_id)
            sl = self.kv.pool.append(r.seq_id, len(f))
            toks += f
            pos += list(range(start, start + len(f)))
            slots += sl
            cu.append(cu[-1] + len(f))
            ctx.append(start + len(f))
            tab = self.kv.pool.block_table(r.seq_id)
            bt[j, :len(tab)] = tab
            lidx.append(cu[-1] - 1)
            max_q = max(max_q, len(f))
            max_ctx = max(max_ctx, start + len(f))
        dev = lambda a, dt: torch.tensor(a, dtype=dt).to(self.device, non_blocking=True)
        enc_starts = dev([r.slot * T_enc for r in live], torch.int32)
        enc_lens = dev([T_enc] * len(live), torch.int32)
        logits = self.model.decode_step(
            dev(toks, torch.int32), dev(pos, torch.int32), dev(slots, torch.int32),
            dev(cu, torch.int32), dev(ctx, torch.int32), dev(bt, torch.int32), max_q, max_ctx,
            self.kv.k, self.kv.v, self.xkv, enc_starts, enc_lens, dev(lidx, torch.int64), self.ws)
        return self._argmax(logits).cpu().numpy()

    # ----------------------------------------------------------- admission
    def _admit(self, reqs: list[STTRequest], slots: list[int],
               device_pcm: torch.Tensor | None = None) -> None:
        """Front end + encoder for newly arrived requests, their cross-attention
        K|V into ``slots``, and their decoder sequences (fed the SOT prompt)."""
        self._encode(reqs, slots, device_pcm)
        self._start_decode(reqs)

    def rows_needed(self, reqs: list[STTRequest]) -> int:
        """Encoder rows / cross-attention slots of ``reqs`` (one per 30 s window)."""
        return sum(n_windows(self._n_samples(r), self.max_windows) for r in reqs)

    @property
    def max_windows(self) -> int:
        return max(1, min(MAX_WINDOWS, self.max_batch))

    def _encode(self, reqs: list[STTRequest], slots: list[int],
                device_pcm: torch.Tensor | None = None) -> None:
        """GPU half of admission (any thread with its own stream): PCM upload,
        log-mel + encoder, cross-attention K|V into the requests' slots (one per
        30 s window, in order); returns once that work is complete (the RMS
        read-back synchronises)."""
        tr = tracer()
        dev = self.device if self.is_gpu else None
        t_enc0 = time.perf_counter()
        with tr.span("h2d", dev, batch=len(reqs)):
            audio, sumsq = self.upload(reqs, device_pcm)
        t0 = time.perf_counter()
        with tr.span("encode", dev, batch=len(reqs)):
            enc = self.encode(audio)
            self.cross_kv(enc, slots)
        ss = sumsq.cpu().numpy()
        if self.is_gpu:
            torch.cuda.current_stream(self.device).synchronize()
        t1 = time.perf_counter()
        self.stats["encode_s"] += t1 - t0
        for r in reqs:
            r.t_enc0, r.t_enc1 = t_enc0, t1
        i = 0
        for r in reqs:
            w = r.windows
            n = max(1, r.n_samples)
            r.sumsq = float(ss[i:i + w].sum())
            r.rms = float(np.sqrt(r.sumsq / n))
            r.slots = list(slots[i:i + w])
            r.slot = r.slots[0]
            i += w

    def _start_decode(self, reqs: list[STTRequest]) -> None:
        """Decoder sequences for encoded requests (scheduler thread)."""
        now = time.perf_counter()
        for r in reqs:
            r.t_dec0 = now
            r.t_done = 0.0
            r.win_texts, r.prev_tokens = [], []
            if not r.slots:
                r.slots = [r.slot]
            self._begin_window(r, 0)

    def _window_text(self, r: STTRequest, w: int) -> str | None:
        """Teacher-forcing text of window ``w`` (None: free decoding)."""
        if r.transcript_windows is not None:
            return r.transcript_windows[w] if w < len(r.transcript_windows) else ""
        if r.transcript is None:
            return None
        if r.windows == 1:
            return r.transcript
        words = r.transcript.split()
        per = -(-len(words) // r.windows)
        return " ".join(words[w * per:(w + 1) * per])

    def _begin_window(self, r: STTRequest, w: int) -> None:
        """A fresh decoder sequence for window ``w`` of ``r`` over its encoder
        rows; later windows are prompted with the previous windows' text."""
        r.win = w
        r.slot = r.slots[w]
        r.seq_id = self._next
        self._next += 1
        self.kv.pool.add_seq(r.seq_id, [])
        prompt = []
        if w > 0 and self.sop is not None and r.prev_tokens and PREV_TOKENS > 0:
            prompt = [self.sop] + r.prev_tokens[-PREV_TOKENS:]
        r.tokens, r.step, r.feed = [], 0, prompt + list(self.sot)
        r.prompt_steps = -(-len(r.feed) // len(self.sot))
        r.target = None
        text = self._window_text(r, w)
        if text is not None:
            room = self.cfg.n_text_ctx - 8 - len(r.feed)
            r.target = self.tok.encode(" " + text.strip())[:room] + [self.eot]

    def _decode_once(self, live: list[STTRequest]) -> list[STTRequest]:
        """One decoder step over ``live`` (at most ``step_tokens`` tokens: a
        sequence may sit the step out or feed only part of its SOT prompt, see
        ``batching.plan_step``); returns the requests that finished."""
        take = plan_step([len(r.feed) for r in live], self.step_tokens, len(self.sot), self._rr)
        self._rr = (self._rr + self.step_tokens) % len(live) if len(live) > self.step_tokens else 0
        step, rest = [], []
        for r, n in zip(live, take):
            if n:
                step.append(r)
                rest.append(r.feed[n:])
                r.feed = r.feed[:n]
        live = step
        nxt = self._step(live)
        self.stats["decode_steps"] += 1
        done = []
        for j, r in enumerate(live):
            if rest[j]:            # part of the prompt still to feed: logits unused
                r.feed = rest[j]
                continue
            t = int(r.target[r.step]) if r.target is not None else int(nxt[j])
            r.tokens.append(t)
            r.step += 1
            if t == self.eot or len(r.tokens) >= r.max_new_tokens or \
                    (r.target is not None and r.step >= len(r.target)):
                f = self._finish(r)
                if f is not None:
                    done.append(f)
            else:
                r.feed = [t]
        return done

    def _finish(self, r: STTRequest) -> STTRequest | None:
        """Window ``r.win`` of ``r`` is decoded: start the next window (None)
        or complete the request (its windows' texts joined)."""
        toks = [x for x in r.tokens if x != self.eot]
        r.win_texts.append(self.tok.decode(toks).strip())
        r.prev_tokens = (r.prev_tokens + toks)[-max(PREV_TOKENS, 1):]
        self.kv.pool.free_seq(r.seq_id)
        if r.win + 1 < r.windows:
            self.stats["long_form_windows"] = self.stats.get("long_form_windows", 0) + 1
            self._begin_window(r, r.win + 1)
            return None
        r.t_done = time.perf_counter()
        r.text = " ".join(t for t in r.win_texts if t)
        self.stats["utterances"] += 1
        return r

    def transcribe(self, reqs: list[STTRequest], device_pcm: torch.Tensor | None = None
                   ) -> list[STTRequest]:
        """Synchronous batch: encode all, decode until every request is done."""
        if not reqs:
            return reqs
        rows = self.rows_needed(reqs)
        assert rows <= self.max_batch, "batch (30 s windows) exceeds max_batch"
        self._admit(reqs, list(range(rows)), device_pcm)
        t_dec = time.monotonic()
        live, steps = list(reqs), 0
        while live:
            self._decode_once(live)
            steps += 1
            live = [r for r in live if r.t_done == 0.0]
        tracer().record("stt_decode", t_dec, time.monotonic(), steps=steps, batch=len(reqs))
        return reqs

    # --------------------------------------------- continuous batching
    def start(self, stream_priority: int = 0) -> None:
        """Start the STT scheduler thread: requests submitted with
        ``submit_batch`` are encoded on arrival and join the RUNNING decoder
        batch at the next step boundary (each in its own cross-attention slot),
        so an utterance never waits for an earlier batch's decode to drain."""
        if getattr(self, "_sched", None) is not None:
            return
        from ..utils.gil import tune_switch_interval
        tune_switch_interval()
        self._inbox: queue.Queue = queue.Queue()
        self._running = True
        self._free_slots = list(range(self.max_batch))
        self._sched = threading.Thread(target=self._schedule, args=(stream_priority,),
                                       name="stt-scheduler", daemon=True)
        self._sched.start()

    def stop(self) -> None:
        if getattr(self, "_sched", None) is None:
            return
        self._running = False
        self._inbox.put(None)
        self._sched.join(timeout=60)
        self._sched = None

    def submit_batch(self, reqs: list[STTRequest], on_done=None) -> Future:
        """Queue requests; ``on_done(req)`` fires on the scheduler thread as
        each finishes; the future resolves with ``reqs`` when all are done."""
        self.start()
        fut: Future = Future()
        if getattr(self, "_fatal", None) is not None:
            fut.set_exception(self._fatal)
            return fut
        reqs = list(reqs)
        if len(reqs) > 1 and self.rows_needed(reqs) > self.max_batch:
            # admission needs a free slot for every window of an inbox item: an
            # oversize batch would wait forever, so it goes in smaller items
            return join_futures([self.submit_batch([r], on_done) for r in reqs], reqs)
        if self.rows_needed(reqs) > self.max_batch:
            fut.set_exception(ValueError(f"utterance needs {self.rows_needed(reqs)} 30 s windows "
                                         f"> max_batch {self.max_batch}"))
            return fut
        self._inbox.put((reqs, on_done, fut))
        return fut

    def _schedule(self, stream_priority: int) -> None:
        try:
            if self.is_gpu:
                from ..utils.streams import placed_stream
                torch.cuda.set_device(self.device)
                torch.cuda.set_stream(placed_stream(self.device, "stt", stream_priority))
                if os.environ.get("LOQA_STT_WAVE_PRIO", "0") == "1":
                    # the latency-bound decoder's waves win issue arbitration
                    # against co-resident LLM GEMM waves (set per thread)
                    ops.set_launch_priority(1)
        except Exception as e:  # noqa: BLE001 - never leave submitters waiting
            self._fatal = e
            while True:
                try:
                    it = self._inbox.get_nowait()
                except queue.Empty:
                    return
                if it is not None and not it[2].done():
                    it[2].set_exception(e)
        live: list[STTRequest] = []
        waiting: list[tuple] = []          # (reqs, cb, fut) not yet admitted (no free slot)
        encoding: list[tuple] = []         # (reqs, future) on the encoder worker
        cells: dict[int, list] = {}
        head_bypass = 0                     # admissions that passed the blocked head
        # the encoder runs on its own worker thread + stream, overlapped with
        # the running decoder batch (an arrival's encode no longer stalls every
        # live transcription); requests join at the next step boundary after
        # their encoder output and cross-attention K|V are complete (inline
        # encodes measured 1.8x slower, docs/PERF.md)
        overlap = self.is_gpu
        enc_pool = self._encoder_executor() if overlap else None
        pl = None
        if self.pipelined:
            from .stt_pipeline import STTPipeline
            pl = STTPipeline(self)
        while self._running:
            idle = not live and not waiting and not encoding
            items = [self._inbox.get()] if idle else []
            while True:
                try:
                    items.append(self._inbox.get_nowait())
                except queue.Empty:
                    break
            for it in items:
                if it is not None:
                    waiting.append(it)
            try:
                new: list[STTRequest] = []
                n_rows = 0
                # FIFO, except that items which fit may pass a head that does
                # not (a long-form utterance waiting for many free slots), at
                # most HOL_BYPASS times per head so it is never starved
                i = 0
                while i < len(waiting):
                    need = self.rows_needed(waiting[i][0])
                    if need > len(self._free_slots) - n_rows:
                        if i == 0 and head_bypass < HOL_BYPASS:
                            i = 1
                            continue
                        if i == 0:
                            break
                        i += 1
                        continue
                    reqs, cb, fut = waiting.pop(i)
                    if i == 0:
                        head_bypass = 0
                    else:
                        head_bypass += 1
                        self.stats["hol_bypass"] = self.stats.get("hol_bypass", 0) + 1
                        if head_bypass >= HOL_BYPASS:
                            i = len(waiting)      # the head goes next
                    n_rows += need
                    if not reqs:
                        fut.set_result(reqs)
                        continue
                    cell = [len(reqs), fut, reqs, cb]
                    cells[id(cell)] = cell
                    for r in reqs:
                        r.on_done = cell
                    new += reqs
                if new:
                    slots = [self._free_slots.pop(0) for _ in range(n_rows)]
                    if enc_pool is not None:
                        encoding.append((new, enc_pool.submit(self._encode, new, slots)))
                    else:
                        self._admit(new, slots)
                        if pl is not None:
                            for r in new:
                                pl.admit(r)
                        live += new
                if encoding:
                    if not live:
                        wait([f for _, f in encoding], timeout=0.002, return_when=FIRST_COMPLETED)
                    still = []
                    for reqs, f in encoding:
                        if f.done():
                            f.result()
                            self._start_decode(reqs)
                            if pl is not None:
                                for r in reqs:
                                    pl.admit(r)
                            live += reqs
                        else:
                            still.append((reqs, f))
                    encoding = still
                if live:
                    finished = pl.pump(live) if pl is not None else self._decode_once(live)
                    for r in finished:
                        self._free_slots += r.slots or [r.slot]
                        self._free_slots.sort()
                        cell = r.on_done
                        if cell[3] is not None:
                            cell[3](r)
                        cell[0] -= 1
                        if cell[0] == 0:
                            cells.pop(id(cell), None)
                            cell[1].set_result(cell[2])
                    live = [r for r in live if r.t_done == 0.0]
            except Exception as e:  # noqa: BLE001 - fail every waiting batch loudly
                # encoder jobs already submitted keep writing cross-attention K|V
                # into their slots: let them finish before any slot is reused
                wait([f for _, f in encoding])
                if pl is not None:
                    pl.abort()
                for cell in list(cells.values()):
                    if not cell[1].done():
                        cell[1].set_exception(e)
                for r in live:
                    self.kv.pool.free_seq(r.seq_id)
                for _, _, fut in waiting:
                    if not fut.done():
                        fut.set_exception(e)
                live, waiting, cells, encoding = [], [], {}, []
                self._free_slots = list(range(self.max_batch))

    def _encoder_executor(self) -> ThreadPoolExecutor:
        if getattr(self, "_enc_pool", None) is None:
            dev = self.device

            def init():
                from ..utils.streams import placed_stream
                torch.cuda.set_device(dev)
                torch.cuda.set_stream(placed_stream(dev, "encoder"))
            self._enc_pool = ThreadPoolExecutor(1, thread_name_prefix="stt-encoder", initializer=init)
        return self._enc_pool
