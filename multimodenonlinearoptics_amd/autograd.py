"""PyTorch autograd over the MI355X engine's adjoints.

``GreensFunction.apply(medium, envelope, poling)`` returns the Green's
matrices (C, S) of a single-mode Chi2PDC medium as complex128 tensors, for a
time-domain pump envelope (complex, length nFreqs) and a per-z-step poling
profile (real, length nZSteps).  Its backward runs the device adjoint (forward
checkpoints of the field, every step when they fit in a quarter of the device
memory, else every few steps with the states between them rebuilt) and returns
dL/d envelope and dL/d poling in torch's complex-gradient convention.

The forward replaces computeGreensFunction (src/_NonlinearMedium.cpp:263-375)
for a Chi2PDC medium (solvers/Chi2PDC.cpp:27-47) after setPump(customPump)
(src/_NonlinearMedium.cpp:207-222) and a per-step poling.

``BatchSignal.apply(medium, inputs, inTimeDomain)`` is batchSignalSimulation of a
Chi3GNLSE medium (src/_FullyNonlinearMedium.hpp:8-11, solvers/Chi3GNLSE.cpp:39-92)
for a [rows, nFreqs] complex128 tensor; its backward runs the device adjoint
(checkpointed forward, segment recomputation) and returns dL/d inputs.
"""
import numpy as np
import torch


def _check_serial(ctx):
    # the medium keeps the checkpoints of its latest forward only
    if ctx.medium.forwardSerial != ctx.serial:
        raise RuntimeError("the medium ran another differentiable forward after this one; its checkpoints are "
                           "gone: run backward before the next forward on the same medium, or use one medium "
                           "per graph")


def _plain(t):
    """t as a detached contiguous complex128 tensor without lazy conjugation or negation,
    so that its memory holds its values."""
    return t.detach().to(torch.complex128).resolve_conj().resolve_neg().contiguous()


def _direct(medium, *tensors):
    """Whether the engine can work on the tensors' own memory: complex128 matrices on the
    medium's device, allocated by the HIP runtime that the engine runs on (a process
    can hold two: torch's own and the system's).  Waits for the pending work on them if so: the
    engine runs on the medium's stream."""
    if not all(t.is_cuda for t in tensors) or not medium.onDevice([t.data_ptr() for t in tensors]):
        return False
    torch.cuda.current_stream(tensors[0].device).synchronize()
    return True


class GreensFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, medium, envelope, poling, ckpt_every=0):
        env = envelope.detach().cpu().numpy().astype(np.complex128)
        pol = poling.detach().cpu().numpy().astype(np.float64)
        medium.setPump(env)
        medium.setPolingProfile(pol)
        n = len(medium.omega)
        C, S = (torch.empty((n, n), dtype=torch.complex128, device=envelope.device) for _ in range(2))
        if _direct(medium, C, S):
            medium.greensForwardDev(C.data_ptr(), S.data_ptr(), False, True, int(ckpt_every))
        else:
            C, S = (torch.from_numpy(a).to(envelope.device) for a in medium.greensForward(False, True, int(ckpt_every)))
        ctx.medium = medium
        ctx.serial = medium.forwardSerial
        ctx.device = envelope.device
        return C, S

    @staticmethod
    def backward(ctx, gC, gS):
        _check_serial(ctx)
        n = len(ctx.medium.omega)
        gC, gS = (torch.zeros((n, n), dtype=torch.complex128, device=ctx.device) if g is None else _plain(g)
                  for g in (gC, gS))
        if gC.shape == gS.shape == (n, n) and _direct(ctx.medium, gC, gS):
            g_env, g_pol = ctx.medium.greensAdjointDev(gC.data_ptr(), gS.data_ptr())
        else:
            g_env, g_pol = ctx.medium.greensAdjoint(gC.cpu().numpy(), gS.cpu().numpy())
        return (None, torch.from_numpy(g_env).to(ctx.device), torch.from_numpy(g_pol).to(ctx.device), None)


class BatchSignal(torch.autograd.Function):
    @staticmethod
    def forward(ctx, medium, inputs, inTimeDomain=True, ckpt_every=0):
        x = _plain(inputs)
        out = torch.empty_like(x)
        if x.dim() == 2 and x.shape[0] > 0 and x.shape[1] == len(medium.omega) and _direct(medium, x, out):
            medium.batchForwardDev(x.data_ptr(), x.shape[0], out.data_ptr(), bool(inTimeDomain), int(ckpt_every))
        else:
            out = torch.from_numpy(medium.batchForward(x.cpu().numpy(), bool(inTimeDomain), int(ckpt_every)))
        ctx.medium = medium
        ctx.serial = medium.forwardSerial
        ctx.device = inputs.device
        ctx.shape = out.shape
        return out.to(inputs.device)

    @staticmethod
    def backward(ctx, g):
        _check_serial(ctx)
        g = _plain(g)
        gin = torch.empty_like(g)
        if g.shape == ctx.shape and _direct(ctx.medium, g, gin):
            ctx.medium.batchAdjointDev(g.data_ptr(), gin.data_ptr())
        else:
            gin = torch.from_numpy(ctx.medium.batchAdjoint(g.cpu().numpy()))
        return None, gin.to(ctx.device), None, None


def band_energy_loss(out_time, omega, lo=5.0, hi=15.0):
    """Spectral energy of the output rows (time domain) in lo <= omega <= hi."""
    F = torch.fft.fft(out_time, dim=-1)
    band = torch.as_tensor((np.asarray(omega) >= lo) & (np.asarray(omega) <= hi), device=out_time.device)
    return (F.abs() ** 2 * band).sum()


def squeezing_loss(S, r=1.5):
    """||S S^T - r I||_F^2 (the differentiable-poling benchmark loss)."""
    n = S.shape[0]
    M = S @ S.transpose(0, 1) - r * torch.eye(n, dtype=S.dtype, device=S.device)
    return (M.abs() ** 2).sum()
