"""One-shot xGMI collectives over peer-mapped HBM (decode TP hot path).

Decode TP payloads are hidden_size bf16 (4-9 KB) — latency-bound, where
an RCCL ring pays 2(world-1) xGMI hops.  The one-shot scheme
(``csrc/xgmi_comm.hip``: every rank pushes its vector to all peers, every
rank reduces locally) is one hop and, crucially, a plain HIP kernel on
the current stream — so the whole TP decode step captures into a
hipGraph with no RCCL-in-graph dependency.

Safety: ``create()`` runs a numerics self-check against
``torch.distributed.all_reduce`` on real hardware; any failure (IPC
unsupported, coherence mismatch, timeout) falls back to RCCL and says
so once.  The device kernel uses a bounded spin: a dead peer sets a
sticky error flag instead of hanging the GPU, and ``check()`` raises on
it at the next host sync point.

The reference has no distributed code at all; this subsystem serves
decode steps sharded over the GPUs of a node (TP=8).
"""

from __future__ import annotations

import os
import struct
from typing import Optional

import torch

from ..ops import hip_ops as ho

MAX_WORLD = 8


class XgmiComm:
    """Peer-mapped one-shot collective communicator (single node)."""

    def __init__(self, rank: int, world: int, device, slot_bytes: int):
        assert 2 <= world <= MAX_WORLD
        self.rank, self.world = rank, world
        self.device = device
        self.slot_bytes = slot_bytes
        total = ho.XC_OFF_DATA + 2 * MAX_WORLD * slot_bytes
        self.base = ho.xc_alloc(total)
        ho.xc_memset(self.base, 0, ho.XC_OFF_DATA)  # header + flags
        self._opened = []

        import torch.distributed as dist
        handle = ho.xc_ipc_handle(self.base)
        objs = [None] * world
        dist.all_gather_object(objs, handle)
        peer_ptrs = []
        for r, h in enumerate(objs):
            if r == rank:
                peer_ptrs.append(self.base)
            else:
                p = ho.xc_ipc_open(h)
                peer_ptrs.append(p)
                self._opened.append(p)
        ho.xc_h2d(self.base, struct.pack(
            "<8Q", *(peer_ptrs + [0] * (MAX_WORLD - world))))
        dist.barrier()

    # ------------------------------------------------------------------
    def _nstripes(self, nbytes: int) -> int:
        return max(1, min(16, nbytes // 8192))

    def all_reduce(self, t: torch.Tensor, spin_limit: int = 5_000_000):
        """In-place sum over all ranks (bf16 or fp32, contiguous).
        Deterministic and rank-identical (fixed summation order)."""
        nbytes = t.numel() * t.element_size()
        mode = (ho.XC_MODE_AR_BF16 if t.dtype == torch.bfloat16
                else ho.XC_MODE_AR_F32)
        ho.xgmi_coll(t.data_ptr(), t.data_ptr(), self.base, self.rank,
                     self.world, nbytes, self.slot_bytes, mode,
                     self._nstripes(nbytes), spin_limit)

    def all_gather_into(self, out: torch.Tensor, t: torch.Tensor,
                        spin_limit: int = 5_000_000):
        """out[world * n] = concat of every rank's t[n] (any dtype)."""
        nbytes = t.numel() * t.element_size()
        assert out.numel() * out.element_size() == nbytes * self.world
        ho.xgmi_coll(out.data_ptr(), t.data_ptr(), self.base, self.rank,
                     self.world, nbytes, self.slot_bytes, ho.XC_MODE_GATHER,
                     self._nstripes(nbytes), spin_limit)

    def fits(self, t: torch.Tensor) -> bool:
        nbytes = t.numel() * t.element_size()
        return (t.is_contiguous() and nbytes % 16 == 0
                and nbytes <= self.slot_bytes
                and t.dtype in (torch.bfloat16, torch.float32))

    def err(self) -> int:
        return struct.unpack("<I", ho.xc_d2h(self.base + ho.XC_OFF_ERR, 4))[0]

    def check(self):
        if self.err():
            raise RuntimeError(
                "xGMI one-shot collective timed out (peer dead or IPC "
                "mapping broken); sticky device error flag set")

    def close(self):
        for p in self._opened:
            try:
                ho.xc_ipc_close(p)
            except Exception:
                pass
        self._opened = []
        if self.base:
            ho.xc_free(self.base)
            self.base = 0

    # ------------------------------------------------------------------
    @classmethod
    def create(cls, rank: int, world: int, device,
               slot_bytes: int) -> Optional["XgmiComm"]:
        """Build + validate a communicator; None on any failure (caller
        falls back to RCCL).  Validation = numerics vs torch.distributed
        on live hardware, so cross-device coherence is PROVEN at init,
        not assumed."""
        if os.environ.get("LLM_XGMI", "1") == "0":
            return None
        import torch.distributed as dist
        if not (dist.is_initialized() and torch.cuda.is_available()):
            return None
        comm = None
        ok = False
        why = ""
        try:
            comm = cls(rank, world, device, slot_bytes)
            # self-check vs torch.distributed.  The reference reduce runs
            # wherever the process-group backend can (RCCL: device;
            # gloo, as in the 2-process-1-GPU CI test: host).
            on_cpu = "nccl" not in str(dist.get_backend()).lower()
            g = torch.Generator(device="cpu").manual_seed(1234 + rank)
            t = (torch.randn(2048, generator=g).to(device)
                 .to(torch.bfloat16).contiguous())
            ref = t.float().cpu() if on_cpu else t.clone()
            dist.all_reduce(ref)
            comm.all_reduce(t, spin_limit=50_000_000)
            s = torch.randn(512, generator=g).to(device).contiguous()
            full = torch.empty(512 * world, device=device)
            reff = torch.empty(512 * world,
                               device="cpu" if on_cpu else device)
            dist.all_gather_into_tensor(reff, s.cpu() if on_cpu else s)
            comm.all_gather_into(full, s, spin_limit=50_000_000)
            torch.cuda.synchronize()
            if comm.err():
                raise RuntimeError("one-shot self-check timed out")
            atol = 6e-2 if on_cpu else 2e-2  # bf16-sum vs fp32-sum ref
            if not torch.allclose(t.float().cpu(), ref.float().cpu(),
                                  atol=atol, rtol=2e-2):
                raise RuntimeError("one-shot all-reduce numerics mismatch")
            if not torch.equal(full.cpu(), reff.cpu()):
                raise RuntimeError("one-shot all-gather mismatch")
            ok = True
        except Exception as e:
            why = f"{type(e).__name__}: {e}"
        # consensus: every rank must agree, or some would one-shot while
        # others ring-reduce (deadlock) — gather the verdicts
        stats = [None] * world
        try:
            dist.all_gather_object(stats, ok)
        except Exception:
            stats = [False] * world
        if all(stats):
            return comm
        if rank == 0:
            print(f"# xGMI one-shot collectives unavailable "
                  f"({why or 'peer rank failed'}); falling back to RCCL",
                  flush=True)
        if comm is not None:
            try:
                comm.close()
            except Exception:
                pass
        return None
