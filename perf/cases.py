"""The work that a user of this framework has it do, as cases that can be timed.

Five kinds of work, each through the entry point that a program calls:

* solve    a frame of a simulation: the preconditioner plan is updated for the frame's image
           and the native solver (FusedPCG, npsd) runs to 1e-6;
* apply    one application of a native plan, z = P(r), as any Krylov loop of one's own calls it;
* predict  the same through the drop-in module (model_predict -> eval_forward), which is how
           programs written for the reference call it in every iteration;
* fwd, bwd one SM block of a training step (smblock3d.forward / .backward);
* train    a whole training pass over one scene: forward, loss, gradients of all parameters.

FP32 is the default of plans, modules and training; BF16 is the fast option of the solver and
of training activations.  One image channel (diag(A)/6) and three ([air, fluid, non-solid])
are the two models whose weights ship with the package.
"""
import math
import os

import torch
import torch.nn.functional as F

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}
SHIFTS = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]


def listed():
    return [
        # the headline workload: 256^3 pillars, BF16 plan, new image every frame
        dict(name="solve_256_bf16", kind="solve", n1=256, n2=256, n3=256, c=1, levels=5, dtype="bf16", level=0.55),
        # the mid-size solve in the default precision
        dict(name="solve_128_fp32", kind="solve", n1=128, n2=128, n3=128, c=1, levels=5, dtype="fp32", level=0.55),
        # the smallest solve in use: launches and latency
        dict(name="solve_64_fp32", kind="solve", n1=64, n2=64, n3=64, c=1, levels=5, dtype="fp32", level=0.7),
        # the default plan at the headline size
        dict(name="apply_256_fp32", kind="apply", n1=256, n2=256, n3=256, c=1, levels=5, dtype="fp32", level=0.55),
        # three channels on a box that is no cube and no power of two
        dict(name="apply_160x96x224_c3", kind="apply", n1=160, n2=96, n3=224, c=3, levels=5, dtype="fp32", level=0.6),
        # the smallest plan: an application is a chain of tiny launches
        dict(name="apply_32_fp32", kind="apply", n1=32, n2=32, n3=32, c=1, levels=3, dtype="fp32", level=0.7),
        # a program written for the reference, with its three-channel model
        dict(name="predict_128_c3", kind="predict", n1=128, n2=128, n3=128, c=3, levels=5, dtype="fp32", level=0.6),
        # level-0 block of the 256^3 training workload, BF16 activations, both directions
        dict(name="fwd_256_bf16", kind="fwd", n1=256, n2=256, n3=256, c=1, batch=1, dtype="bf16", level=0.65),
        dict(name="bwd_256_bf16", kind="bwd", n1=256, n2=256, n3=256, c=1, batch=1, dtype="bf16", level=0.65),
        # a block on an odd crop with three channels and a batch of right-hand sides
        dict(name="fwd_97x75x131_c3", kind="fwd", n1=97, n2=75, n3=131, c=3, batch=2, dtype="fp32", level=0.6),
        # level-0 block of the default (FP32) training: two right-hand sides a scene
        dict(name="bwd_128_fp32", kind="bwd", n1=128, n2=128, n3=128, c=1, batch=2, dtype="fp32", level=0.6),
        # a training pass of the default training at its default size
        dict(name="train_128_fp32", kind="train", n1=128, n2=128, n3=128, c=1, levels=5, batch=2, dtype="fp32",
             level=0.6),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _dims(rng, volume, step, lo, hi):
    """Three extents, multiples of step, with about the given volume."""
    side = volume ** (1 / 3)
    a, b = (math.exp(rng.uniform(-0.4, 0.4)) for _ in range(2))
    out = [min(hi, max(lo, round(s / step) * step)) for s in (side * a, side * b, side / (a * b))]
    rng.shuffle(out)
    return dict(n1=out[0], n2=out[1], n3=out[2])


def draw(rng):
    """One more case: kinds as often as the listed ones, sizes over the logarithm of the range,
    channels, precisions, batches and water levels as programs use them."""
    kind = rng.choice(["solve", "solve", "apply", "apply", "apply", "predict", "fwd", "fwd", "bwd", "bwd", "train"])
    level = round(rng.uniform(0.4, 0.8), 3)
    c = rng.choice([1, 1, 3])
    if kind == "solve":
        dtype = rng.choice(["fp32", "bf16"])
        top = 6e6 if dtype == "bf16" else 2.5e6
        return dict(kind=kind, c=1, levels=5, dtype=dtype, level=level, **_dims(rng, _log_uniform(rng, 2.6e5, top), 32, 64, 256))
    if kind in ("apply", "predict"):
        levels = rng.choice([3, 4, 5])
        return dict(kind=kind, c=c, levels=levels, dtype="fp32", level=level,
                    **_dims(rng, _log_uniform(rng, 3.3e4, 7e6 if kind == "apply" else 3e6), 1 << levels, 32, 256))
    if kind == "train":
        return dict(kind=kind, c=1, levels=4, batch=rng.choice([1, 2]), dtype="fp32", level=level,
                    **_dims(rng, _log_uniform(rng, 2.6e5, 2.1e6), 16, 48, 160))
    # blocks: any extents; half of them those of a level of a power-of-two grid
    step = rng.choice([1, 64])
    dims = _dims(rng, _log_uniform(rng, 3e4 if step == 1 else 2.6e5, 4e6 if c == 1 else 2e6), step, 17 if step == 1 else 64, 256)
    return dict(kind=kind, c=c, batch=rng.choice([1, 1, 2, 4]), dtype=rng.choice(["fp32", "bf16"]), level=level, **dims)


# ------------------------------------------------------------------ inputs

def _grid(case):
    return case["n1"], case["n2"], case["n3"]


def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * salt + seed)


def _flags(case, seed):
    """Cell flags on the GPU: walls, solid vertical pillars (radius 4 to 10, on a lattice with
    jitter, so that gaps stay open), air above the water level (0 wall, 1 solid, 2 fluid,
    3 air).  Every fluid column reaches the air, so A is regular."""
    n1, n2, n3 = _grid(case)
    f = torch.full((n1, n2, n3), 2, dtype=torch.int8, device="cuda")
    g = torch.Generator().manual_seed(seed)
    i = torch.arange(n1, device="cuda").view(n1, 1)
    j = torch.arange(n2, device="cuda").view(1, n2)
    for a in range(24, n1 - 23, 48):
        for b in range(24, n2 - 23, 48):
            u = torch.rand(3, generator=g).tolist()
            r = 4 + 6 * u[0]
            f[(i - a - 8 * u[1]) ** 2 + (j - b - 8 * u[2]) ** 2 <= r * r] = 1
    air = min(int(case["level"] * n3), n3 - 3)
    top = f[:, :, air + 1:]
    top[top == 2] = 3
    for d in range(3):
        f.select(d, 0).fill_(0)
        f.select(d, f.shape[d] - 1).fill_(0)
    return f


def _shifted(x, d):
    """x[..., v + d], zero outside the grid."""
    n = x.shape[-3:]
    p = F.pad(x, (1, 1, 1, 1, 1, 1))
    return p[..., 1 + d[0]:1 + d[0] + n[0], 1 + d[1]:1 + d[1] + n[1], 1 + d[2]:1 + d[2] + n[2]]


def _faces(x):
    return [_shifted(x, d) for d in SHIFTS if abs(d[0]) + abs(d[1]) + abs(d[2]) == 1]


def _image(flags, c):
    """One channel: diag(A)/6 on the fluid; three: [air, fluid, non-solid]."""
    if c == 1:
        open_ = (flags >= 2).float()
        return (sum(_faces(open_)) / 6 * (flags == 2))[None].contiguous()
    return torch.stack([flags == 3, flags == 2, flags >= 2]).float()


def _rhs(flags, count, seed):
    b = torch.randn(count, *flags.shape, generator=_gen(seed, 1), device="cuda") * (flags == 2)
    return b / b.flatten(1).norm(dim=1).view(-1, 1, 1, 1)


def _weights(case, seed):
    """Weights and bias of one block as the modules draw them."""
    c, bound = case["c"], (27 * case["c"]) ** -0.5
    w = torch.rand(27, c, 3, 3, 3, generator=_gen(seed, 2), device="cuda") * 2 - 1
    b = torch.rand(27, generator=_gen(seed, 3), device="cuda") * 2 - 1
    return w * bound, b * bound


def _state_dict(case):
    """The package's trained weights where they fit; None (the module's own seeded draw) for
    other depths and for training, which starts from it."""
    import mlpcg_amd
    if case["levels"] != 5 or case["kind"] == "train":
        return None
    path = os.path.join(os.path.dirname(mlpcg_amd.__file__), "weights", f"sm_l5_c{case['c']}.pt")
    return torch.load(path, map_location="cuda", weights_only=True)


def _model(case):
    from mlpcg_amd.sm_model_3d import SmallSMModelDn3D
    torch.manual_seed(7)
    m = SmallSMModelDn3D(case["levels"], case["c"], "trilinear").to("cuda")
    sd = _state_dict(case)
    if sd is not None:
        m.load_state_dict(sd)
    return m


def _block_inputs(case, seed):
    """Image of the scene, activations, and an upstream gradient of a mean-of-squares loss."""
    dt = DTYPES[case["dtype"]]
    flags = _flags(case, seed)
    shape = (case["batch"], 1, *_grid(case))
    x = torch.randn(shape, generator=_gen(seed, 4), device="cuda").to(dt)
    g = (1e-2 * torch.randn(shape, generator=_gen(seed, 5), device="cuda")).to(dt)
    w, b = _weights(case, seed)
    return _image(flags, case["c"]).to(dt), x, g, w, b


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fwd", "bwd"):
        image, x, g, w, b = _block_inputs(case, seed)
        return dict(kind=kind, image=image, x=x, g=g, w=w, b=b)
    flags = _flags(case, seed if kind != "predict" else 0)  # predict: one scene, its cells are the unknowns
    model = _model(case)
    if kind == "train":
        from mlpcg_amd.scenes import Scene
        from mlpcg_amd.train import SceneBatch
        sb = SceneBatch(Scene(flags.cpu().numpy(), seed, "pillars"), case["c"], torch.device("cuda"))
        return dict(kind=kind, model=model, sb=sb, cache=sb.model_input(model, DTYPES[case["dtype"]]),
                    rhs=_rhs(flags, case["batch"], seed).flatten(1))
    image = _image(flags, case["c"])
    r = _rhs(flags, 1, seed)[0]
    if kind == "predict":
        from mlpcg_amd.solver import model_predict
        cells = (flags.flatten() == 2).nonzero().flatten()
        return dict(kind=kind, predict=model_predict(model, image, cells), r=r.flatten()[cells])
    plan = model.make_preconditioner(image, DTYPES[case["dtype"]])
    if kind == "apply":
        return dict(kind=kind, plan=plan, r=r)
    from mlpcg_amd.solver import FusedPCG
    return dict(kind=kind, plan=plan, image=image, solver=FusedPCG(flags.cpu().numpy()), b=r.flatten())


def run(state):
    kind = state["kind"]
    if kind == "solve":
        state["plan"].update(state["image"])
        return state["solver"].solve(state["b"], state["plan"], method="npsd", max_it=300, tol=1e-6)[0]
    if kind == "apply":
        return state["plan"].apply(state["r"])
    if kind == "predict":
        return state["predict"](state["r"])
    if kind == "train":
        from mlpcg_amd.train import relative_residual_sq_dot
        model, sb, rhs = state["model"], state["sb"], state["rhs"]
        x = model.forward_cached(state["cache"], rhs.view(rhs.shape[0], 1, *sb.shape))
        loss = relative_residual_sq_dot(sb, x, rhs)
        grads = torch.autograd.grad(loss, list(model.parameters()))
        return [loss.detach(), torch.cat([g.flatten() for g in grads])]  # one bucket, as for an all-reduce
    from mlpcg_amd.sm_model_3d import smblock3d
    if kind == "fwd":
        return smblock3d.forward(state["image"], state["x"], state["w"], state["b"])
    return smblock3d.backward(state["g"], state["image"], state["x"], state["w"], state["b"])


# ------------------------------------------------------------------ necessary work

def _iterations(case):
    """About how many iterations npsd takes here with the shipped weights."""
    return 10 + 0.25 * (case["n1"] * case["n2"] * case["n3"]) ** (1 / 3)


def work(case):
    v, c = case["n1"] * case["n2"] * case["n3"], case["c"]
    s = 2 if case["dtype"] == "bf16" else 4
    stencil, dot = 2 * 27 * (27 * c + 1) * v, 2 * 27 * v  # K of every voxel; its product with x
    if case["kind"] == "fwd":
        return dict(bytes=s * v * (c + 2 * case["batch"]), flops=stencil + case["batch"] * dot)
    if case["kind"] == "bwd":  # dx (K and its transpose), the outer products and their contraction
        return dict(bytes=s * v * (c + 3 * case["batch"]), flops=2 * stencil + 2 * case["batch"] * dot)
    pyramid = sum(8.0 ** -l for l in range(case["levels"]))
    model = 2 * pyramid * (stencil + dot)
    if case["kind"] in ("apply", "predict"):
        return dict(bytes=(4 * c + 8) * v, flops=model)
    if case["kind"] == "train":
        b = case["batch"]
        return dict(bytes=(4 * c + 12 * b) * v, flops=2 * pyramid * (3 * stencil + 3 * b * dot))
    it = _iterations(case)  # an iteration: r in and z out of P, the direction and the residual updates
    return dict(bytes=it * 54 * v, flops=it * (model + 60 * v))


# ------------------------------------------------------------------ values in 64 bits

def _patches(x):
    """(..., 27, V): the 27 neighbours of every cell."""
    return torch.stack([_shifted(x, d).flatten(-3) for d in SHIFTS], dim=-2)


def _block64(image, x, w, b):
    """y[b, v] = sum_p K_p(v) x[b, v + d_p], K = W patches(image) + b."""
    k = w.reshape(27, -1) @ _patches(image).flatten(0, 1) + b.reshape(27, 1)
    return torch.stack([(k * _patches(xi[0])).sum(0).view(xi.shape) for xi in x])


def _coef64(image, w, b):
    v = image[0].numel()
    ybar = torch.stack([torch.stack([_shifted(ch, d).sum() for d in SHIFTS]) for ch in image]) / v
    return (w.flatten() * ybar.flatten()).sum() + b


def _model64(sd, levels, image, x):
    imgs = [image]
    for _ in range(levels):
        imgs.append(F.avg_pool3d(imgs[-1][None], 2)[0])
    down = [_block64(imgs[0], x, sd["pre.0.weight"], sd["pre.0.bias"])]
    for i in range(1, levels + 1):
        name = f"pre.{i}" if i < levels else "l"
        down.append(_block64(imgs[i], F.avg_pool3d(down[-1], 2), sd[name + ".weight"], sd[name + ".bias"]))
    up = down[levels]
    for i in range(levels - 1, -1, -1):
        up = F.interpolate(up, scale_factor=2, mode="trilinear")
        up = _block64(imgs[i], up, sd[f"post.{i}.weight"], sd[f"post.{i}.bias"])
        up = (_coef64(imgs[i], sd[f"c0.{i}.weight"], sd[f"c0.{i}.bias"]) * down[i]
              + _coef64(imgs[i], sd[f"c1.{i}.weight"], sd[f"c1.{i}.bias"]) * up)
    return up


def _laplacian(flags):
    """x -> A x on the full grid for x that vanishes off the fluid."""
    fluid = (flags == 2).double()
    diag = sum(_faces((flags >= 2).double())) * fluid
    return lambda x: diag * x - sum(_faces(x)) * fluid


def _solution(flags, b):
    """A^-1 b by conjugate gradients (diagonal scaling) far below the tolerance of the solves."""
    apply, x, r = _laplacian(flags), torch.zeros_like(b), b.clone()
    scale = (flags == 2) / sum(_faces((flags >= 2).double())).clamp(min=1)
    z = scale * r
    p, rz, stop = z.clone(), (r * z).sum(), float(b.norm()) * 1e-11
    for k in range(4000):
        ap = apply(p)
        a = rz / (p * ap).sum()
        x += a * p
        r -= a * ap
        z = scale * r
        rz, old = (r * z).sum(), rz
        p = z + rz / old * p
        if k % 50 == 49 and float(r.norm()) < stop:
            break
    return x


def exact(case, seed):
    kind, levels = case["kind"], case.get("levels")
    if kind in ("fwd", "bwd"):
        image, x, g, w, b = (t.double() for t in _block_inputs(case, seed))
        if kind == "fwd":
            return [_block64(image, x, w, b)]
        for t in (x, w, b):
            t.requires_grad_()
        return list(torch.autograd.grad(_block64(image, x, w, b), (x, w, b), g))
    flags = _flags(case, seed if kind != "predict" else 0)
    image = _image(flags, case["c"]).double()
    if kind == "solve":
        return _solution(flags, _rhs(flags, 1, seed)[0].double()).flatten()
    model = _model(case)
    sd = {k: v.detach().double() for k, v in model.state_dict().items()}
    if kind == "train":
        for v in sd.values():
            v.requires_grad_()
        b = _rhs(flags, case["batch"], seed).double()
        x = _model64(sd, levels, image, b[:, None])[:, 0] * (flags == 2)
        a = _laplacian(flags)
        loss = torch.stack([((bi - a(xi)) ** 2).sum() / (bi ** 2).sum() for bi, xi in zip(b, x)]).mean()
        grads = torch.autograd.grad(loss, [sd[k] for k, _ in model.named_parameters()])
        return [loss.detach(), torch.cat([g.flatten() for g in grads])]
    r = _rhs(flags, 1, seed)
    if kind == "apply":
        return _model64(sd, levels, image, r[None].double())[0, 0]
    cells = (flags.flatten() == 2).nonzero().flatten()
    b = torch.zeros(flags.numel(), dtype=torch.float64, device="cuda")
    b[cells] = (r.flatten()[cells].double() / r.flatten()[cells].double().norm())
    return _model64(sd, levels, image, b.view(1, 1, *_grid(case))).flatten()[cells]
