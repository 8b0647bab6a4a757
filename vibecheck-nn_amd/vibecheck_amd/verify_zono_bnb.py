"""Batched bound primitives on the GPU (HIP library), with the reference's
function names and signatures (verify_zono_bnb.py of the reference).

Every function takes the reference's ``gg`` dict (fc / relu / conv /
reshape ops, and the constant add / sub / mul and residual-merge add ops)
and fp32 GPU tensors, computes with the kernels of
libvibecheck_amd.so, and returns new tensors.  Unsupported ops raise
NotImplementedError, fp64 raises NotImplementedError, CPU tensors raise
RuntimeError: there is no other compute path.
"""
import ctypes

import torch

from . import _lib, mlp_fused
from ._lib import call, f32, host_array, ptr, stream

__all__ = ['_make_slopes', '_ibp_forward_graph_batched',
           '_forward_zonotope_graph_batched', '_crown_intermediate_batched',
           '_spec_backward_graph_batched',
           '_run_alpha_crown_inputsplit_batched']

# Use the whole-network kernels for narrow fc/ReLU chains (<= 64 wide).
# Switching this off routes those nets through the layer-wise kernels.
FUSED_MLP = True
# Fuse a relu relaxation into the conv backward after it where the conv
# qualifies (vc_backward_relu_conv); off: the relu is applied on its own.
FUSED_RELU_CONV = True


def _plan(gg, dev):
    return mlp_fused.plan_for(gg, dev) if FUSED_MLP else None


def _zono_sb(gg, xl, xh, device, dtype):
    """Zonotope pre-activation bounds only (the fused kernel when the net
    qualifies, else the layer-wise forward)."""
    plan = _plan(gg, xl.device)
    if plan is not None:
        sb, _ = mlp_fused.zono_bounds(
            plan, xl, xh,
            lambda a, b: _forward_zonotope_graph_batched(a, b, gg, device, dtype)[0])
        return sb
    return _zono_forward(xl, xh, gg, dtype, True)[0]


def _check_dtype(dtype):
    if dtype is not None and dtype != torch.float32:
        raise NotImplementedError(
            f'vibecheck_amd computes in fp32 only, got {dtype}')


# --------------------------------------------------------------------------
# Device copies of the network parameters, cached on the gg dict
# --------------------------------------------------------------------------

def _op_params(op, device):
    """fp32 contiguous device copies of an op's tensors (cached on the op,
    like the reference caches converted biases on op dicts,
    verify_zono_bnb.py:4482-4486)."""
    key = '_vc_amd_params'
    cached = op.get(key)
    if cached is not None and cached['device'] == device:
        return cached
    p = {'device': device, 'name': op['name']}
    if op['type'] == 'fc':
        p['W'] = op['W'].detach().to(device=device, dtype=torch.float32).contiguous()
        b = op.get('bias')
        p['b'] = (None if b is None else
                  torch.as_tensor(b).detach().to(device=device, dtype=torch.float32)
                  .reshape(-1).contiguous())
        p['n_out'], p['n_in'] = p['W'].shape
    elif op['type'] == 'conv':
        k = op['kernel'].detach().to(device=device, dtype=torch.float32).contiguous()
        if k.dim() != 4:
            raise NotImplementedError('vibecheck_amd: conv kernels must be 4-D')
        p['K'] = k
        b = op.get('bias')
        p['b'] = (None if b is None else
                  torch.as_tensor(b).detach().to(device=device, dtype=torch.float32)
                  .reshape(-1).contiguous())
        C_in, H, W = op['in_shape']
        C_out, Ho, Wo = op['out_shape']
        kh, kw = k.shape[2], k.shape[3]
        sh, sw = _pair(op['stride'])
        ph, pw = _pair(op['padding'])
        p['geom'] = (C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo)
        p['n_in'] = C_in * H * W
        p['n_out'] = C_out * Ho * Wo
    # the caller's own fp32 tensors are as ready as the caller has them; copies
    # are ready for every stream before they are kept
    given = (op.get('W', op.get('kernel')), op.get('bias'))
    made = [p.get('W', p.get('K')), p.get('b')]
    own = all(t is None or torch.is_tensor(g) and g.data_ptr() == t.data_ptr()
              for t, g in zip(made, given))
    if own or _lib.settled(device):
        op[key] = p
    return p


def _prod(shape):
    n = 1
    for s in shape:
        n *= int(s)
    return n


def _fc_form(op, width):
    """How an fc reads a node of ``width`` values per domain: (P, nd_out).

    P = 1 is the plain form, width == W.shape[1].  The N-D batched MatMul
    form (an ONNX MatMul on a (prefix..., n_in) input,
    verify_zono_bnb.py:3145-3168 and 4382-4401) has in_shapes_nd[0] with
    two or more dims, W.shape[1] equal to its last and width equal to its
    product: W applies to each of the P = prod(prefix) slices of n_in
    values, and the output holds P slices of W.shape[0].  nd_out tells
    whether the op also carries the out_shape_nd the reference's backward
    needs for that form (two or more dims).  Any other width raises
    ValueError: the kernels would read a wider tensor as rows of
    W.shape[1]."""
    n_out, n_in = (int(s) for s in op['W'].shape)
    shp = (op.get('in_shapes_nd') or [None])[0]
    if shp is not None and len(shp) >= 2 and int(shp[-1]) == n_in \
            and width == _prod(shp):
        P = _prod(shp[:-1])
        shp_o = op.get('out_shape_nd')
        nd_out = shp_o is not None and len(shp_o) >= 2 and _prod(shp_o) == P * n_out
        return P, nd_out
    if width == n_in:
        return 1, True
    raise ValueError(f'fc {op["name"]!r}: input of {width} values per domain, but W is '
                     f'{n_out}x{n_in} and in_shapes_nd is {shp}')


def validate_gg(gg, n_in=None):
    """The width of every node of ``gg``, checked op by op from the input's
    (``n_in``, else gg['input_n'], else the product of gg['input_shape']
    past the batch dim) before any launch, with the ops' shapes only (no
    device tensors): an fc reads W.shape[1] values or the N-D MatMul form
    (_fc_form); a conv reads prod(in_shape) and writes prod(out_shape); a
    residual merge adds two nodes of one width; relu, reshape and the
    constant add / sub / mul keep the width.  Raises ValueError on the
    first mismatch, NotImplementedError on an op type outside
    fc / conv / relu / reshape / add / sub / mul.  Returns {name: width}."""
    if n_in is None:
        n_in = gg.get('input_n')
        if n_in is None:
            shp = gg.get('input_shape')
            if shp is None:
                raise ValueError('gg has neither input_n nor input_shape')
            n_in = _prod(shp[1:]) if len(shp) > 1 else _prod(shp)
    width = {gg['input_name']: int(n_in)}
    for op in gg['ops']:
        t, name = op['type'], op['name']
        for i in op['inputs']:
            if i not in width:
                raise ValueError(f'{t} {name!r}: input {i!r} is not computed before it')
        w = width[op['inputs'][0]]
        if t == 'fc':
            P, _ = _fc_form(op, w)
            width[name] = P * int(op['W'].shape[0])
        elif t == 'conv':
            want = _prod(op['in_shape'])
            if w != want:
                raise ValueError(f'conv {name!r}: input of {w} values per domain, '
                                 f'in_shape {tuple(op["in_shape"])} holds {want}')
            width[name] = _prod(op['out_shape'])
        elif t == 'add' and op.get('is_merge'):
            w2 = width[op['inputs'][1]]
            if w2 != w:
                raise ValueError(f'add {name!r}: merges widths {w} and {w2}')
            width[name] = w
        elif t in ('relu', 'reshape', 'add', 'sub', 'mul'):
            width[name] = w
        else:
            _unsupported('validate_gg', op)
    return width


def _widths(gg, n_in):
    """validate_gg for a call on inputs of n_in values per domain, cached on
    the gg for its op list and input width."""
    key = (id(gg['ops']), len(gg['ops']), int(n_in))
    hit = gg.get('_vc_amd_widths')
    if hit is not None and hit[0] == key:
        return hit[1]
    w = validate_gg(gg, n_in)
    gg['_vc_amd_widths'] = (key, w)
    return w


class _Packs:
    """The weights in the layouts that one call's products read.  Each is made
    on first use, on the call's stream, from the weights as they are then, and
    goes with the call: another thread's call on its own stream packs for
    itself, and a weight written between two calls (also through ``.data``,
    which no version counter shows) is seen by the second.  1024 x 1024 weights
    take 6 us, of products of 100 us and more; a launch takes 5 whatever it
    packs, so the first need of a layout makes it of every layer of the network
    that the same rule takes."""

    def __init__(self, gg, dev):
        self.gg, self.dev, self._made = gg, dev, {}

    def _params(self, kind):
        return [_op_params(op, self.dev) for op in self.gg['ops'] if op['type'] == kind]

    def _make(self, entry, keys, params, describe, dtype, st):
        """One launch: the weights of ``params`` into buffers under ``keys``;
        ``describe`` gives their sizes and the host arrays of the layers' shapes,
        which the graph keeps by those shapes."""
        shapes = self.gg.setdefault('_vc_amd_packs', {})
        at = (entry, *keys, *[q.get('geom', (q['n_in'], q['n_out'])) for q in params])
        if at not in shapes:
            sizes, rows = describe()
            shapes[at] = (sizes, sum(sizes), sum(rows, []) if len(keys) == 1 else
                          [host_array(ctypes.c_int32, r) for r in rows])
        sizes, total, arrays = shapes[at]
        out = torch.empty(total, dtype=dtype, device=self.dev)
        if len(keys) == 1:
            q = params[0]
            call(entry, ptr(q['W'] if 'W' in q else q['K']), *arrays, ptr(out), st)
            self._made[keys[0]] = out
            return
        outs = out.split(sizes)
        src, src_p = host_array(ctypes.c_void_p,
                                [ptr(q['W'] if 'W' in q else q['K']) for q in params])
        dst, dst_p = host_array(ctypes.c_void_p, [ptr(o) for o in outs])
        call(entry + '_many', src_p, *[p for _, p in arrays], dst_p, len(keys), st)
        self._made.update(zip(keys, outs))

    def fc(self, p, st, trans=False, others=()):
        """The bf16 parts of an fc's W, or of its transpose; ``others``: (params,
        transposed) that the call will need as well."""
        if (p['name'], trans) not in self._made:
            want = [(p, trans)] + [q for q in others if q[0] is not p or q[1] != trans]
            want = [(q, t) for q, t in want if (q['name'], t) not in self._made]

            def describe():
                KN = [(q['n_in'], q['n_out']) if t else (q['n_out'], q['n_in']) for q, t in want]
                size = _lib.load().vc_fc_split_pack_bytes
                return ([size(K, N) for K, N in KN],
                        [[K for K, _ in KN], [N for _, N in KN], [int(t) for _, t in want]])
            self._make('vc_fc_split_pack', [(q['name'], t) for q, t in want],
                       [q for q, _ in want], describe, torch.uint8, st)
        return self._made[p['name'], trans]

    def conv_interval(self, p, K, st):
        """The parts of a conv's kernel and of its magnitudes for
        vc_ibp_conv_split."""
        out = self._made.get((p['name'], 'interval'))
        if out is None:
            n = p['K'].shape[0]
            out = [torch.empty(_lib.load().vc_fc_split_pack_bytes(K, n), dtype=torch.uint8,
                               device=p['K'].device) for _ in range(2)]
            call('vc_fc_split_pack_abs', ptr(p['K']), K, n, 1, ptr(out[0]), ptr(out[1]), st)
            self._made[p['name'], 'interval'] = out
        return out

    def has_taps(self, p, window):
        return (p['name'], 'taps', window) in self._made

    def conv_taps(self, p, st, window=False):
        """A conv kernel's transposed taps by output-parity class
        (vc_conv_t_pack); ``window``: without the padding, for rows that carry
        their place in the image."""
        key = (p['name'], 'taps', window)
        if key not in self._made:
            # the fold kernel's convs, of up to four channels, take none
            want = [p] + [q for q in self._params('conv')
                          if q is not p and q['geom'][0] > 4 and not self.has_taps(q, window)]

            def describe():
                geom, sizes = [], []
                for q in want:
                    C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = q['geom']
                    geom += [C_out, C_in, kh, kw, sh, sw] + ([0, 0] if window else [ph, pw])
                    sizes.append(_lib.load().vc_conv_t_pack_floats(C_out, C_in, kh, kw, sh, sw))
                    if sizes[-1] < 0:
                        raise RuntimeError(f'vc_conv_t_pack_floats: bad geometry {q["geom"]}')
                return sizes, [geom]
            # rows of four floats: every buffer starts on 16 bytes
            self._make('vc_conv_t_pack', [(q['name'], 'taps', window) for q in want], want,
                       describe, torch.float32, st)
        return self._made[key]

    def _conv_split_pays(self, p, M, R, shared):
        last = p.get('split_pays')  # of the rows asked for last
        if last is None or last[0] != (M, R, shared):
            C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
            bands = 0 if _few_channels(p) else _lib.load().vc_backward_conv_split_fits(
                M, R, 1 if shared else 0, C_out, Ho, Wo, C_in, H, W, kh, kw, sh, sw, ph, pw)
            last = (M, R, shared), (
                bands == 1 or bands > 1 and (M >= _CONV_SPLIT_ROWS or M * p['n_out'] * C_in * kh
                                             * kw >= _CONV_SPLIT_MACS))
            p['split_pays'] = last
        return last[1]

    def conv_split(self, p, M, R, shared, st):
        """A conv kernel's bf16 parts for vc_backward_conv_split of M rows (R a
        domain, shared by all domains or not); None where the geometry or the
        rows are outside that kernel, or the fp32 product is the faster one."""
        if not self._conv_split_pays(p, M, R, shared):
            return None
        key = (p['name'], 'conv_split')
        if key not in self._made:
            want = [p] + [q for q in self._params('conv')
                          if q is not p and (q['name'], 'conv_split') not in self._made
                          and self._conv_split_pays(q, M, R, shared)]

            def describe():
                geom = [[q['geom'][i] for i in (3, 0, 4, 5, 6, 7)] for q in want]
                return ([_lib.load().vc_conv_split_pack_bytes(*g) for g in geom],
                        [sum(geom, [])])
            self._make('vc_conv_split_pack', [(q['name'], 'conv_split') for q in want], want,
                       describe, torch.uint8, st)
        return self._made[key]


def _few_channels(p, window=None):
    """Whether a conv (of windows: (rows' height and width, the result's)) is the
    fold kernel's: a few input channels, the network's first layer."""
    key = ('fold_ok', window)
    if key not in p:
        C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
        if window is not None:
            (Ho, Wo, H, W), ph, pw = window, 0, 0
        p[key] = bool(_lib.load().vc_backward_relu_conv_ok(C_out, Ho, Wo, C_in, H, W, kh, kw,
                                                           sh, sw, ph, pw))
    return p[key]


def _fc_split_pays(M, K, N, once, sweep):
    """Whether M rows of K values times (K, N) are the faster as parts: ``once``,
    packed for one pass; ``sweep``, a gradient sweep follows that uses the
    backward's slopes (the figures stand at _FC_SPLIT_WIDTH)."""
    if K < _TWO_PHASE_MIN_WIDTH or max(K, N) < _FC_SPLIT_WIDTH:
        return False
    # the parts of wide rows for few columns, written and read again, have to
    # stay in the last-level cache
    if K > _TWO_PHASE_MIN_WIDTH and (4 * N >= K or 6 * M * K <= 288 << 20):
        if M >= 8192 or (M >= 4096 if once else M >= 2048) and M * K * N >= (1e9 if once else 4e8):
            return True
    return sweep and _FC_SPLIT_SWEEP_ROWS <= M < 8192 and (K <= 512 or M >= 2048)


def _fc_split_parts(packs, p, M, st, trans=False, once=False, sweep=False):
    """The fc weights' bf16 parts for M rows' vc_backward_fc_split (``trans``:
    for the gradient's products with W^T); None where the fp32 product is the
    faster one."""
    def pays(q, t):
        if t:
            return M >= _FC_SPLIT_SWEEP_ROWS and min(q['n_in'], q['n_out']) >= _FC_SPLIT_WIDTH
        return _fc_split_pays(M, q['n_out'], q['n_in'], once, sweep)
    if M >= 1 << 31 or not pays(p, trans):
        return None
    if (p['name'], trans) in packs._made:
        return packs.fc(p, st, trans)
    forms = (True,) if trans else (False, True) if sweep else (False,)
    return packs.fc(p, st, trans, [(q, t) for q in packs._params('fc') for t in forms
                                   if pays(q, t)])


def _cut(t, rows):
    return t if t is None or rows is None else t[rows]


def _in_slices(B, R, K, dev, launch):
    """``launch`` a vc_fc_split product of B * R rows of K values, in slices whose
    parts take up to _FC_WORK_BYTES: whole domains, or rows of one domain.  It
    gets the slice (for _cut) of a (B, ..), a (B * R, ..) and a shared (R, ..)
    tensor, its number of rows and of rows a domain, and the buffer of parts."""
    size = _lib.load().vc_fc_split_pack_bytes
    most = max(64, _FC_WORK_BYTES // (size(K, 16) // 16))
    if B * R <= most:
        launch(None, None, None, B * R, R,
               torch.empty(size(K, B * R), dtype=torch.uint8, device=dev))
        return
    if R <= most:
        step = -(-B // -(-B // (most // R)))  # the slices alike
        spans = [(b, min(B, b + step), 0, R) for b in range(0, B, step)]
    else:
        step = -(-R // -(-R // most))
        spans = [(b, b + 1, r, min(R, r + step)) for b in range(B) for r in range(0, R, step)]
    rows = max((b1 - b0) * (r1 - r0) for b0, b1, r0, r1 in spans)
    work = torch.empty(size(K, rows), dtype=torch.uint8, device=dev)
    for b0, b1, r0, r1 in spans:
        launch(slice(b0, b1), slice(b0 * R + r0, (b1 - 1) * R + r1), slice(r0, r1),
               (b1 - b0) * (r1 - r0), r1 - r0, work)


def _pair(v):
    if isinstance(v, int):
        return v, v
    v = tuple(int(x) for x in v)
    return (v[0], v[0]) if len(v) == 1 else (v[0], v[1])


def _unsupported(fn, op):
    raise NotImplementedError(
        f'{fn}: unsupported op {op["type"]!r} at {op["name"]!r} -- silently '
        f'skipping would certify unsound bounds')


# --------------------------------------------------------------------------
# add / sub / mul: their constants, and residual merges
# --------------------------------------------------------------------------

def _op_const(op, key, device, n):
    """An add/sub op's 'bias' or a mul op's 'scale' as an fp32 device
    vector of n values, or of one value for a scalar (None when the op has
    none).  The reference converts the float64 constant with
    torch.as_tensor(..., dtype=float32) and broadcasts it against the n
    values: a vector of the trailing N-D dimension repeats along the
    leading ones (out_shape_nd, verify_zono_bnb.py:3240-3251, 4490-4503);
    a mul's per-channel vector repeats over each channel's H x W
    (in_shapes_nd, :3523-3534, :4702-4708).  Cached on the op."""
    cached = op.get('_vc_amd_' + key)
    if cached is not None and cached[0] == (str(device), n):
        return cached[1]
    v = op.get(key)
    if v is None:
        return None
    t = torch.as_tensor(v, dtype=torch.float32).reshape(-1).cpu()
    k = t.numel()
    if k not in (1, n):
        shp_in = (op.get('in_shapes_nd') or [None])[0]
        shp_out = op.get('out_shape_nd')
        if (key == 'scale' and shp_in is not None and len(shp_in) == 3
                and int(shp_in[0]) == k and k * int(shp_in[1]) * int(shp_in[2]) == n):
            t = t.repeat_interleave(int(shp_in[1]) * int(shp_in[2]))
        elif shp_out is not None and len(shp_out) >= 1 and int(shp_out[-1]) == k and n % k == 0:
            t = t.repeat(n // k)
        else:
            raise ValueError(f'{op["type"]} {op["name"]!r}: {key} of {k} values does not '
                             f'broadcast to {n}')
    t = t.to(device).contiguous()
    op['_vc_amd_' + key] = ((str(device), n), t)
    return t


def _fork_points(gg):
    """The names consumed by more than one op (the gg's 'fork_points',
    network.py:1713; derived from the ops when the dict has none)."""
    fp = gg.get('fork_points')
    if fp is not None:
        return fp
    uses = {}
    for op in gg['ops']:
        for i in op['inputs']:
            uses[i] = uses.get(i, 0) + 1
    return {k for k, v in uses.items() if v > 1}


def _shared_gens(name_a, name_b, gg, gen_count):
    """Generator columns two merging branches share: the count at the first
    fork point among name_a's ancestors (depth-first from name_a, inputs
    pushed in order) that is also an ancestor of name_b, else at the input.
    The reference's _find_shared_gens_count (verify_zono_bnb.py:2387-2428);
    column k of every descendant of a fork is that fork's k-th noise."""
    forks = _fork_points(gg)
    pred = {op['name']: op['inputs'] for op in gg['ops']}

    def ancestors(name):
        order, stack, seen = [], [name], set()
        while stack:
            x = stack.pop()
            if x in seen:
                continue
            seen.add(x)
            order.append(x)
            stack.extend(pred.get(x, ()))
        return order

    anc_b = set(ancestors(name_b))
    for a in ancestors(name_a):
        if a in anc_b and a in forks:
            return gen_count.get(a, 0)
    return gen_count.get(gg['input_name'], 0)


# --------------------------------------------------------------------------
# a1: ReLU relaxation
# --------------------------------------------------------------------------

def _make_slopes(lo, hi):
    """CROWN adaptive slopes (verify_zono_bnb.py:503-522).

    Returns (lo_s, up_s, up_t, active, dead, unstable) like the reference.
    """
    lo, hi = f32(lo), f32(hi)
    if lo.shape != hi.shape:
        raise ValueError('lo/hi shape mismatch')
    outs = [torch.empty_like(lo) for _ in range(3)]
    masks = [torch.empty(lo.shape, dtype=torch.bool, device=lo.device)
             for _ in range(3)]
    call('vc_make_slopes', ptr(lo), ptr(hi), lo.numel(),
         *[ptr(t) for t in outs], *[ptr(t) for t in masks], stream())
    return (*outs, *masks)


# --------------------------------------------------------------------------
# a2: IBP forward
# --------------------------------------------------------------------------

def _ibp_forward_graph_batched(xl, xh, gg, device, dtype, relu_clamps=None,
                               root_sb=None):
    """Batched interval forward (verify_zono_bnb.py:1066-1153).

    Returns {layer_idx: (lo, hi)} of (B, n_L) pre-activation bounds after
    root intersection, split clamps and crossing repair.
    """
    _check_dtype(dtype)
    xl, xh = f32(xl), f32(xh)
    B = xl.shape[0]
    dev = xl.device
    widths = _widths(gg, xl.shape[1])
    lo = {gg['input_name']: xl}
    hi = {gg['input_name']: xh}
    sb = {}
    st = stream()
    packs = _Packs(gg, dev)
    # nodes without a relu below them: their intervals are exact, CROWN's first
    # bounds equal them up to rounding and choose slopes by the larger of the
    # two, so their sums keep their order
    raw = {gg['input_name']}
    for op in gg['ops']:
        t = op['type']
        name = op['name']
        if t != 'relu' and all(i in raw for i in op['inputs']):
            raw.add(name)
        l, h = lo[op['inputs'][0]], hi[op['inputs'][0]]
        if t == 'fc':
            if _fc_form(op, widths[op['inputs'][0]])[0] > 1:
                # the reference's interval fc is mid @ W.T (verify_zono_bnb.py:
                # 1108-1113), which has no N-D MatMul form
                raise NotImplementedError(
                    f'_ibp_forward_graph_batched: fc {name!r} is an N-D batched MatMul, '
                    f'which the interval forward does not take')
            p = _op_params(op, dev)
            lo_o = torch.empty(B, p['n_out'], device=dev)
            hi_o = torch.empty_like(lo_o)
            slices = _lib.load().vc_ibp_fc_slices(B, p['n_in'], p['n_out'])
            if slices > 1:
                work = torch.empty(slices * B * p['n_out'] * 2, dtype=torch.float64, device=dev)
                call('vc_ibp_fc_sliced', ptr(l), ptr(h), B, p['n_in'], ptr(p['W']), ptr(p['b']),
                     p['n_out'], ptr(lo_o), ptr(hi_o), slices, ptr(work), st)
            else:
                call('vc_ibp_fc', ptr(l), ptr(h), B, p['n_in'], ptr(p['W']),
                     ptr(p['b']), p['n_out'], ptr(lo_o), ptr(hi_o), st)
            lo[name], hi[name] = lo_o, hi_o
        elif t == 'conv':
            p = _op_params(op, dev)
            C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
            lo_o = torch.empty(B, p['n_out'], device=dev)
            hi_o = torch.empty_like(lo_o)
            K = C_in * kh * kw
            per = 2 * _lib.load().vc_fc_split_pack_bytes(K, Ho * Wo)
            if (name not in raw and K >= 512 and C_out > 32
                    and B * p['n_out'] * K >= _IBP_SPLIT_MACS
                    and per <= _IBP_BOX_BYTES and H * W < 1 << 28 and p['n_in'] < 1 << 31):
                parts = packs.conv_interval(p, K, st)
                work = torch.empty(per * max(1, min(B, _ZONO_WORK_BYTES // per)),
                                   dtype=torch.uint8, device=dev)
                call('vc_ibp_conv_split', ptr(l), ptr(h), B, C_in, H, W, ptr(parts[0]),
                     ptr(parts[1]), ptr(p['b']), C_out, kh, kw, sh, sw, ph, pw, Ho, Wo,
                     ptr(lo_o), ptr(hi_o), ptr(work), work.numel(), st)
            else:
                call('vc_ibp_conv', ptr(l), ptr(h), B, C_in, H, W, ptr(p['K']),
                     ptr(p['b']), C_out, kh, kw, sh, sw, ph, pw, Ho, Wo,
                     ptr(lo_o), ptr(hi_o), st)
            lo[name], hi[name] = lo_o, hi_o
        elif t == 'relu':
            L = op.get('layer_idx')
            n = l.shape[1]
            rlo = rhi = cl = ch = None
            if L is not None and root_sb is not None and L in root_sb:
                rlo = f32(root_sb[L][0]).reshape(-1)
                rhi = f32(root_sb[L][1]).reshape(-1)
            if L is not None and relu_clamps is not None and L in relu_clamps:
                cl = f32(relu_clamps[L][0])
                ch = f32(relu_clamps[L][1])
            sl = torch.empty_like(l)
            sh_ = torch.empty_like(l)
            pl = torch.empty_like(l)
            ph_ = torch.empty_like(l)
            call('vc_ibp_relu', ptr(l), ptr(h), B, n, ptr(rlo), ptr(rhi),
                 ptr(cl), ptr(ch), ptr(sl), ptr(sh_), ptr(pl), ptr(ph_), st)
            if L is not None:
                sb[L] = (sl, sh_)
            lo[name], hi[name] = pl, ph_
        elif t == 'reshape':
            lo[name], hi[name] = l, h
        elif t == 'add' and op.get('is_merge'):
            # residual merge (verify_zono_bnb.py:1133-1135)
            l2, h2 = lo[op['inputs'][1]], hi[op['inputs'][1]]
            lo_o, hi_o = torch.empty_like(l), torch.empty_like(h)
            call('vc_add_ew', ptr(l), ptr(l2), l.numel(), ptr(lo_o), st)
            call('vc_add_ew', ptr(h), ptr(h2), h.numel(), ptr(hi_o), st)
            lo[name], hi[name] = lo_o, hi_o
        elif t in ('add', 'sub'):
            # constant shift (verify_zono_bnb.py:1136-1143)
            n = l.shape[1]
            b = _op_const(op, 'bias', dev, n)
            if b is None:
                raise ValueError(f'{t} {name!r}: no constant')
            mode = 0 if t == 'add' else 1
            lo_o, hi_o = torch.empty_like(l), torch.empty_like(h)
            call('vc_affine_ew', ptr(l), B, n, 1, ptr(b), b.numel(), mode, ptr(lo_o), st)
            call('vc_affine_ew', ptr(h), B, n, 1, ptr(b), b.numel(), mode, ptr(hi_o), st)
            lo[name], hi[name] = lo_o, hi_o
        elif t == 'mul':
            # constant scale (verify_zono_bnb.py:1144-1148)
            n = l.shape[1]
            s = _op_const(op, 'scale', dev, n)
            if s is None:
                raise ValueError(f'mul {name!r}: no scale')
            lo_o, hi_o = torch.empty_like(l), torch.empty_like(h)
            call('vc_interval_mul', ptr(l), ptr(h), B, n, ptr(s), s.numel(), ptr(lo_o),
                 ptr(hi_o), st)
            lo[name], hi[name] = lo_o, hi_o
        else:
            raise NotImplementedError(
                f'_ibp_forward_graph_batched: unsupported op {t!r} at '
                f'{name!r} -- silently skipping would certify unsound bounds')
    return sb


# --------------------------------------------------------------------------
# a3: zonotope forward
# --------------------------------------------------------------------------

def _forward_zonotope_graph_batched(xl, xh, gg, device, dtype):
    """Batched zonotope forward (verify_zono_bnb.py:3079-4075, fc/relu/conv/
    reshape/add/sub/mul).  Returns (sb, (c, G)); G is (B, n, K) with the new
    generator columns of each ReLU padded to the batch maximum, as in the
    reference; a residual merge sums the generator columns the two branches
    share from their fork point and appends each branch's own.
    (The (c, G) output needs the layer-wise kernels; bound-only callers use
    the fused kernel through _zono_sb.)
    """
    sb, out = _zono_forward(xl, xh, gg, dtype, False)
    _forward_zonotope_graph_batched.last_bilinear_op_bounds = {}
    return sb, out


class _Gens:
    """Generators whose form a following fc uses: ``lists`` (idx, idx_ld, mu,
    xl, xh, cnt, k) for columns that are one neuron's, after the columns ``G``
    (B, n, K) scaled by ``lam`` (B, n); ``dense`` gives the (B, n, K + k) matrix."""
    __slots__ = ('G', 'lam', 'lists', 'dense')

    def __init__(self, G, lam, lists, dense):
        self.G, self.lam, self.lists, self.dense = G, lam, lists, dense


def _zono_fc(packs, p, g, B, K, st):
    """(B, n_out, K + k) generators of a _Gens through an fc."""
    idx, idx_ld, mu, xl, xh, cnt, k = g.lists
    n, n_out, dev = p['n_in'], p['n_out'], p['W'].device
    out = torch.empty(B, n_out, K + k, device=dev)
    if K:
        parts = packs.fc(p, st, True)
        size = _lib.load().vc_fc_split_pack_bytes
        per = size(n, K)
        work = torch.empty(per * min(B, _ZONO_WORK_BYTES // per) if per <= _ZONO_WORK_BYTES
                           else max(size(n, 64), _ZONO_WORK_BYTES), dtype=torch.uint8, device=dev)
        call('vc_zono_fc_split', ptr(g.G), ptr(g.lam), B, n, K, ptr(parts), n_out, K + k,
             ptr(out), ptr(work), work.numel(), st)
    call('vc_zono_fc_cols', ptr(p['W']), n_out, n, B, k, ptr(idx), idx_ld, ptr(mu), ptr(xl),
         ptr(xh), ptr(cnt), K, K + k, ptr(out), st)
    return out


def _zono_forward(xl, xh, gg, dtype, bounds_only):
    """(sb, (c, G) of the last op); with ``bounds_only`` fc layers above the
    last relu are left out and the second is None."""
    _check_dtype(dtype)
    xl, xh = f32(xl), f32(xh)
    B, n_in = xl.shape
    dev = xl.device
    st = stream()
    widths = _widths(gg, n_in)
    varying = ((xh - xl) / 2).abs().amax(dim=0) > 0 if B > 0 else \
        torch.zeros(n_in, dtype=torch.bool, device=dev)
    vidx = varying.nonzero(as_tuple=True)[0].to(torch.int32).contiguous()
    K = int(vidx.numel())
    ops = gg['ops']
    packs = _Packs(gg, dev)
    users = {}
    for op in ops:
        for i in op['inputs']:
            users.setdefault(i, []).append(op)
    top = max([i for i, op in enumerate(ops) if op['type'] == 'relu' and 'layer_idx' in op],
              default=len(ops))
    if not bounds_only or any(op['type'] not in ('fc', 'reshape') for op in ops[top + 1:]):
        top = len(ops)

    def one_fc(name):
        """The fc that alone reads a node, in its plain form, or None."""
        u = users.get(name, [])
        if len(u) == 1 and u[0]['type'] == 'fc' and _fc_form(u[0], widths[name])[0] == 1:
            return u[0]
        return None

    def input_dense():
        G = torch.empty(B, n_in, K, device=dev)
        call('vc_zono_input', ptr(xl), ptr(xh), B, n_in, ptr(vidx), K, ptr(c), ptr(G), st)
        return G

    c = torch.empty(B, n_in, device=dev)
    if one_fc(gg['input_name']) is not None and B > 0:
        call('vc_zono_input', ptr(xl), ptr(xh), B, n_in, ptr(vidx), 0, ptr(c), None, st)
        G = _Gens(None, None, (vidx, 0, None, xl, xh, None, K), input_dense)
    else:
        G = input_dense()
    state = {gg['input_name']: (c, G)}
    gen_count = {gg['input_name']: K}
    sb = {}
    for pos, op in enumerate(ops):
        t = op['type']
        name = op['name']
        c_in, G_in = state[op['inputs'][0]]
        Kc = gen_count[op['inputs'][0]]
        if isinstance(G_in, _Gens) and t != 'fc':
            G_in = G_in.dense()
        n = c_in.shape[1]
        if t == 'add' and op.get('is_merge'):
            # residual merge: the fork point's generators are shared
            # (verify_zono_bnb.py:3213-3234)
            c_b, G_b = state[op['inputs'][1]]
            Kb = G_b.shape[2]
            shared = _shared_gens(op['inputs'][0], op['inputs'][1], gg, gen_count)
            if not (0 <= shared <= Kc and shared <= Kb):
                raise ValueError(f'add {name!r}: {shared} shared generators of {Kc} and {Kb}')
            c_o = torch.empty_like(c_in)
            call('vc_add_ew', ptr(c_in), ptr(c_b), c_in.numel(), ptr(c_o), st)
            G_o = torch.empty(B, n, Kc + Kb - shared, device=dev)
            call('vc_zono_merge', ptr(G_in), Kc, ptr(G_b), Kb, shared, B * n, ptr(G_o), st)
            state[name] = (c_o, G_o)
        elif t in ('add', 'sub'):
            # constant shift of the centre (verify_zono_bnb.py:3235-3265)
            b = _op_const(op, 'bias', dev, n)
            c_o = c_in
            if b is not None:
                c_o = torch.empty_like(c_in)
                call('vc_affine_ew', ptr(c_in), B, n, 1, ptr(b), b.numel(),
                     0 if t == 'add' else 1, ptr(c_o), st)
            state[name] = (c_o, G_in)
        elif t == 'mul':
            # constant scale of centre and generators (verify_zono_bnb.py:3501-3536)
            s = _op_const(op, 'scale', dev, n)
            if s is None:
                raise ValueError(f'mul {name!r}: no scale')
            c_o = torch.empty_like(c_in)
            call('vc_affine_ew', ptr(c_in), B, n, 1, ptr(s), s.numel(), 2, ptr(c_o), st)
            G_o = torch.empty_like(G_in)
            if Kc > 0:
                call('vc_affine_ew', ptr(G_in), B, n, Kc, ptr(s), s.numel(), 2, ptr(G_o), st)
            state[name] = (c_o, G_o)
        elif t == 'fc':
            p = _op_params(op, dev)
            # the N-D MatMul form (verify_zono_bnb.py:3145-3168) applies W to
            # each of P slices: (B, P * n_in) centres and (B, P * n_in, K)
            # generators are (B * P, n_in) and (B * P, n_in, K) as they lie
            P, _ = _fc_form(op, widths[op['inputs'][0]])
            c_o = torch.empty(B, P * p['n_out'], device=dev)
            if isinstance(G_in, _Gens):
                call('vc_zono_fc', ptr(c_in), None, B, p['n_in'], 0, ptr(p['W']), ptr(p['b']),
                     p['n_out'], ptr(c_o), None, st)
                k = G_in.lists[-1]
                state[name] = (c_o, _zono_fc(packs, p, G_in, B, Kc - k, st))
                gen_count[name] = Kc
                continue
            G_o = torch.empty(B, P * p['n_out'], Kc, device=dev)
            call('vc_zono_fc', ptr(c_in), ptr(G_in), B * P, p['n_in'], Kc,
                 ptr(p['W']), ptr(p['b']), p['n_out'], ptr(c_o), ptr(G_o), st)
            state[name] = (c_o, G_o)
        elif t == 'conv':
            p = _op_params(op, dev)
            C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
            c_o = torch.empty(B, p['n_out'], device=dev)
            G_o = torch.empty(B, p['n_out'], Kc, device=dev)
            call('vc_zono_conv', ptr(c_in), ptr(G_in), B, Kc, C_in, H, W,
                 ptr(p['K']), ptr(p['b']), C_out, kh, kw, sh, sw, ph, pw, Ho,
                 Wo, ptr(c_o), ptr(G_o), st)
            state[name] = (c_o, G_o)
        elif t == 'relu':
            n = c_in.shape[1]
            lo = torch.empty(B, n, device=dev)
            hi = torch.empty_like(lo)
            rank = torch.empty(B, n, dtype=torch.int32, device=dev)
            cnt = torch.empty(B, dtype=torch.int32, device=dev)
            call('vc_zono_relu_bounds', ptr(c_in), ptr(G_in), B, n, Kc,
                 ptr(lo), ptr(hi), ptr(rank), ptr(cnt), st)
            if 'layer_idx' in op:
                sb[op['layer_idx']] = (lo, hi)
            if pos == top:
                return sb, None
            nxt = one_fc(name)
            together = (nxt is not None
                        and B * n * Kc * int(nxt['W'].shape[0]) >= _ZONO_SPLIT_MACS)
            if together and Kc:
                # queued before the host waits, with those of the layers to come
                # (generators only grow in number)
                packs.fc(_op_params(nxt, dev), st, True,
                         [(_op_params(v, dev), True) for v in map(
                             one_fc, (o['name'] for o in ops[pos + 1:top] if o['type'] == 'relu'))
                          if v is not None and B * Kc * int(v['W'].numel()) >= _ZONO_SPLIT_MACS])
            k_new = int(cnt.max().item()) if B > 0 else 0
            c_o = torch.empty(B, n, device=dev)
            if together:
                lam = torch.empty(B, n, device=dev)
                idx = torch.empty(B, max(k_new, 1), dtype=torch.int32, device=dev)
                mu = torch.empty(B, max(k_new, 1), device=dev)
                call('vc_zono_relu_lists', ptr(c_in), ptr(lo), ptr(hi), ptr(rank), B, n, k_new,
                     ptr(c_o), ptr(lam), ptr(idx), ptr(mu), st)
                G_o = _Gens(G_in, lam, (idx, k_new, mu, None, None, cnt, k_new), None)
            else:
                G_o = torch.empty(B, n, Kc + k_new, device=dev)
                call('vc_zono_relu_apply', ptr(c_in), ptr(G_in), ptr(lo), ptr(hi),
                     ptr(rank), B, n, Kc, k_new, ptr(c_o), ptr(G_o), st)
            state[name] = (c_o, G_o)
            gen_count[name] = Kc + k_new
            continue
        elif t == 'reshape':
            state[name] = (c_in, G_in)
        else:
            raise ValueError(f'batched zono forward: unknown op type {t!r}')
        gen_count[name] = state[name][1].shape[2]
    return sb, state[ops[-1]['name']]


# --------------------------------------------------------------------------
# a5-a8: CROWN backward + concretization
# --------------------------------------------------------------------------

class _Rows:
    """Backward coefficient rows at one graph node.

    ``ew`` is (R, n) when ``shared`` (identical for every domain, before the
    first per-domain relaxation) else (B*R, n).  ``relu`` names a relu layer
    whose relaxation is still to be applied (it is fused into the next fc).
    ``alpha``/``beta`` belong to that pending relu; ``alpha_group`` (B,)
    int64 makes ``alpha`` (G*R, n) the rows of each domain's group.
    ``window`` (a _Window) says that ``ew`` holds only that part of each row's
    image, the rest being zero.
    """
    __slots__ = ('ew', 'shared', 'relu', 'alpha', 'alpha_row', 'beta', 'alpha_group',
                 'n_groups', 'window')

    def __init__(self, ew, shared):
        self.ew = ew
        self.shared = shared
        self.relu = None
        self.alpha = None
        self.alpha_row = 0
        self.beta = None
        self.alpha_group = None
        self.n_groups = 0
        self.window = None


class _Window:
    """Rows (.., C, wh, ww) at ``origin`` (R, 2) of (C, H, W) images: what a
    few conv neurons' rows meet of the layers below them."""
    __slots__ = ('origin', 'wh', 'ww', 'C', 'H', 'W')

    def __init__(self, origin, wh, ww, C, H, W):
        self.origin, self.wh, self.ww, self.C, self.H, self.W = origin, wh, ww, C, H, W

    def worth(self):
        """Windows up to half of the image are carried as such: beyond, the
        part outside the image and the wider steps cost what is saved.  Images
        of more than 2^30 values are past the window kernels' offsets."""
        return (2 * self.wh * self.ww <= self.H * self.W
                and self.C * self.H * self.W <= 1 << 30)


# A zonotope relu and fc are taken together from this many multiplications up:
# below, the few more launches cost what the product saves (forwards of three
# layers, apart and together: 784-256x3-10 of 16 boxes, 0.8e9 in the second
# layer, 327 and 341 us; of 64 boxes, 3.3e9, 605 and 531).  Parts take so many
# bytes at a time, which the last-level cache holds.
_ZONO_SPLIT_MACS = 1.5e9
# The interval forward of a conv likewise: the pass that forms its parts writes
# 12 bytes per pixel and tap whatever the channels out.  The gathering product
# and the parts, weights packed included, us (values K of a pixel -> channels):
#   512 -> 33    0.07e9 multiplications 55 and 34, 4.7e9 1,290 and 774
#   512 -> 128   0.08e9 52 and 37, 1.2e9 216 and 76;  576 -> 64  0.15e9 44 and 34
#   1600 -> 33   0.05e9 111 and 61, 14e9 3,072 and 2,585
# and from 512 values and 33 channels on they win everywhere but 1600 -> 64 at
# 1.7e9 (151 and 154).  Onto 16 channels they lose from
# 0.3e9 up (576: 1.9 times at 0.6e9, 1024: 1.5 at 5e9).  With fewer values they
# win from 0.6e9 up only (288 -> 33 0.85, 128 -> 64 0.6 of the time; below, 1.2 to
# 1.8 times): left with the gathering product.
_IBP_SPLIT_MACS = 1e8
_ZONO_WORK_BYTES = 192 << 20
_IBP_BOX_BYTES = 1 << 30  # parts of one box: beyond, the gathering product, which takes none


class BackwardTrace:
    """Per-relu stored pre-relaxation rows of one backward, for the alpha
    gradient sweep: entries (L, P, p_shared) in backward order.  ``other``
    names an op the sweep does not replay (add, sub, mul, a fan-in); ``slopes``
    holds the layers' slopes where the backward had to form them and they are
    small (_SLOPES_KEPT_BYTES; for one row a domain they are three times the
    rows): beyond, the sweep forms them again."""

    def __init__(self):
        self.relus = []
        self.fcs = []
        self.slopes = {}
        self.other = None


# vc_backward_fc runs as relaxation pass + plain MFMA GEMM from this row
# width up when given a relaxed-rows buffer (measured 2x faster on 1024-wide
# layers than relaxing inside the GEMM's loads).
_TWO_PHASE_MIN_WIDTH = 64

# Products of bf16 parts against the fp32 ones, both from the rows to the product,
# us; the parts also take 6 for the slopes and, once a call, 5.5 to pack the
# weights.  Backward, (values x columns) at rows:
#   64 x 128      2,304: 14 and 10;  73,728: 30 and 34 (a single tile's width in fp32)
#   65 x 128     18,432: 44 and 27;  73,728: 107 and 60
#   128 x 128     4,608: 17 and 11;   9,216: 27 and 15;  73,728: 105 and 48
#   256 x 256       288: 15 and 10;   4,608: 22 and 18;  13,824: 85 and 29
#   512 x 512       576: 15 and 14;   2,304: 30 and 25;   4,608: 47 and 32
#   784 x 128     4,608: 41 and 32;  36,864: 182 and 137; 73,728: 250 and 248
#   1024 x 784    1,152: 32 and 34;   2,304: 48 and 42;   4,608: 79 and 67
#   1024 x 64     2,304: 29 and 26;  18,432: 115 and 75;  73,728: 290 and 286
#   1024 x 1024     288: 20 and 26;   2,304: 75 and 48;  73,728: 1,202 and 991
# The gradient's, whose fp32 product sums in 64 bits (slopes on both sides):
#   128 x 128       288: 10 and 9;  256 x 256: 15 and 10;  1024 x 1024: 52 and 25;
#   128 x 33     18,432: 18 and 18;  64 x 64: 10 and 14.
_FC_SPLIT_SWEEP_ROWS = 64
_FC_SPLIT_WIDTH = 128
# The split conv takes a large image band by band in one workgroup, a few rows of
# them on as many CUs, while the gathering product spreads their pixels.  Both
# from the rows to the product, weights packed, us (split; relu and fp32 conv):
#   16 -> 8, 3x3, 28x28    6 rows 65 and 37;  60: 65 and 56;  120: 65 and 70
#   33 -> 17, 3x3, 20x20   6: 76 and 47;     120: 78 and 71;  300: 97 and 112
#   64 -> 64, 3x3, 32x32   6 (0.23e9 multiplications): 210 and 153;  12: 212 and
#                          195;  30 (1.1e9): 213 and 239
# An image in one band is as fast or faster at any number of rows (13 -> 8, 14x14,
# 6: 22 and 25; 64 -> 32, 4x4 stride 2 onto 32x32, 6: 51 and 48, 12: 52 and 57).
_CONV_SPLIT_ROWS = 128
_CONV_SPLIT_MACS = 5e8
# Below, packing the taps costs what it saves (with it and without: 16 -> 8,
# 28x28, 60 rows 57 and 56, 300 rows 110 and 123; 64 -> 64 onto 16x16, 12 rows 32
# and 31) and is a launch more.
_CONV_TAPS_MACS = 5e7
_SLOPES_KEPT_BYTES = 32 << 20  # a layer's; forming them takes 10 us at that size
# Parts of rows take so much at a time, whatever the number of rows.  Slices
# that the last-level cache holds (192 MiB) are no faster (73,728 rows of 1024 x
# 1024 977 us whole, 991; of 1024 x 64 286 and 312).
_FC_WORK_BYTES = 512 << 20


def _expand_rows(t, B):
    """(R, n) shared rows -> (B*R, n) per-domain rows."""
    R, n = t.shape
    return t.unsqueeze(0).expand(B, R, n).reshape(B * R, n).contiguous()


def _backward(tight, xl, xh, gg, seed_name, seed, seed_shared, acc0,
              alpha_at_layer=None, relu_split_beta=None, trace=None, split=True,
              packs=None, fresh=False):
    """Walk the ops backward from ``seed_name`` and concretize.

    seed: (R, n) rows when ``seed_shared`` else (B*R, n), or a _Rows; acc0:
    (R,) when shared else (B*R,).  split: products may run as bf16 parts on
    the matrix cores; off where the bounds choose slopes, whose step at 1/2
    turns a last-bit change of a bound into another lower slope (on 512 boxes
    through 1024-wide layers one run in four).  packs: the caller's _Packs, where
    it makes several of these calls; fresh: acc0 is this call's to write to.
    Returns (lb (B, R), A, a_shared, acc (B*R,));
    A of window rows is None.
    """
    once = packs is None
    B, n_in = xl.shape
    dev = xl.device
    packs = _Packs(gg, dev) if once else packs
    st = stream()
    widths = _widths(gg, n_in)
    rows = seed if isinstance(seed, _Rows) else _Rows(seed, seed_shared)
    R = rows.ew.shape[0] if seed_shared else rows.ew.shape[0] // max(B, 1)
    acc, acc_own = (acc0, fresh) if seed_shared else (acc0.clone(), True)
    acc_shared = seed_shared
    ew_at = {seed_name: rows}
    ops = gg['ops']

    def per_domain_acc():
        nonlocal acc, acc_own, acc_shared
        if acc_shared:
            if B == 1:  # the expansion is the same memory
                own_acc()
            acc = acc.unsqueeze(0).expand(B, R).reshape(B * R).contiguous()
            acc_own, acc_shared = True, False

    def own_acc():
        """Before a write to shared constant terms: acc0 stays as it is."""
        nonlocal acc, acc_own
        if not acc_own:
            acc, acc_own = acc.clone(), True

    def combine(a, b):
        """Rows reaching one node from two consumers, summed (ew_at[inp] +
        ew, verify_zono_bnb.py:4462-4469)."""
        a, b = materialize(a), materialize(b)
        if a.shared and b.shared:
            out = torch.empty_like(a.ew)
            call('vc_add_ew', ptr(a.ew), ptr(b.ew), a.ew.numel(), ptr(out), st)
            return _Rows(out, True)
        per_domain_acc()
        ea = _expand_rows(a.ew, B) if a.shared else a.ew
        eb = _expand_rows(b.ew, B) if b.shared else b.ew
        out = torch.empty_like(ea)
        call('vc_add_ew', ptr(ea), ptr(eb), ea.numel(), ptr(out), st)
        return _Rows(out, False)

    def put(inp, rows):
        prev = ew_at.get(inp)
        if prev is not None and trace is not None:
            trace.other = trace.other or 'fan-in'
        ew_at[inp] = rows if prev is None else combine(prev, rows)

    def bias_dot(rows, v, sign):
        """acc += sign * rows . v (the constant of an add or sub)."""
        n = rows.ew.shape[1]
        if rows.shared and acc_shared:
            own_acc()
            call('vc_rows_bias_dot', ptr(rows.ew), R, R, n, 1, ptr(v), v.numel(), sign,
                 ptr(acc), st)
        else:
            per_domain_acc()
            call('vc_rows_bias_dot', ptr(rows.ew), B * R, R, n, 1 if rows.shared else 0,
                 ptr(v), v.numel(), sign, ptr(acc), st)

    def bias_acc(rows, p):
        """The bias and the constant terms that a product of rows without a
        pending relu adds rows . bias to.  Shared rows add it once, to shared
        terms; where another branch has given every domain its own by then, it
        is added to all of them here and the product adds none."""
        if rows.shared:
            if not acc_shared:
                if p['b'] is not None:
                    bias_dot(rows, p['b'].repeat_interleave(p['n_out'] // p['b'].numel()), 1.0)
                return None, None
            if p['b'] is not None:
                own_acc()
        else:
            per_domain_acc()
        return p['b'], acc

    def dense(rows):
        """Window rows as whole images (other rows as they are)."""
        w = rows.window
        if w is not None:
            N = rows.ew.shape[0]
            out = torch.empty(N, w.C * w.H * w.W, device=dev)
            call('vc_patch_dense', ptr(rows.ew), ptr(w.origin), N, R, w.C, w.H, w.W, w.wh, w.ww,
                 ptr(out), st)
            rows.ew, rows.window = out, None
        return rows

    def materialize(rows):
        """Apply a pending relu relaxation with the standalone kernel."""
        rows = dense(rows)
        if rows.relu is None:
            return rows
        if rows.alpha_group is not None:
            raise NotImplementedError(
                'vibecheck_amd: group-indexed alpha is supported before an fc only')
        L = rows.relu
        lo, hi = tight[L]
        lo, hi = f32(lo), f32(hi)
        n = lo.shape[1]
        ew = _expand_rows(rows.ew, B) if rows.shared else rows.ew
        per_domain_acc()
        if trace is not None:
            trace.relus.append((L, rows.ew, rows.shared))
        out = torch.empty(B * R, n, device=dev)
        call('vc_backward_relu', ptr(ew), B * R, R, n, ptr(lo), ptr(hi),
             ptr(rows.alpha), rows.alpha_row, ptr(rows.beta), ptr(out),
             ptr(acc), st)
        return _Rows(out, False)

    def conv_fp32(p, ew, M, window, out, bias, acc):
        """M rows through a conv in fp32, acc += rows . bias; the fold kernel
        reads the kernel as it lies, the gathering product its packed taps, or
        for few rows their kernel (the same bits)."""
        C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
        if window is not None:
            (Ho, Wo, H, W), ph, pw = window, 0, 0
        geom = (C_out, Ho, Wo, C_in, H, W, kh, kw, sh, sw, ph, pw)
        if _few_channels(p, window) or (M * C_out * Ho * Wo * C_in * kh * kw < _CONV_TAPS_MACS
                                       and not packs.has_taps(p, window is not None)):
            call('vc_backward_conv', ptr(ew), M, ptr(p['K']), ptr(bias), *geom, ptr(out),
                 ptr(acc), st)
        else:
            call('vc_backward_conv_packed', ptr(ew), M, ptr(p['K']),
                 ptr(packs.conv_taps(p, st, window is not None)), ptr(bias), *geom, ptr(out),
                 ptr(acc), st)

    def slopes(rows):
        """The pending relu's slopes per (domain, neuron) for a conv that
        relaxes its rows as it loads them."""
        lo, hi = f32(tight[rows.relu][0]), f32(tight[rows.relu][1])
        n = lo.shape[1]
        per_domain_acc()
        if trace is not None:
            trace.relus.append((rows.relu, rows.ew, rows.shared))
        out = [torch.empty(B, n, device=dev) for _ in range(3)]
        call('vc_relax_slopes', ptr(lo), ptr(hi), ptr(rows.alpha), B * n, ptr(out[0]),
             ptr(out[1]), ptr(out[2]), st)
        if trace is not None and 12 * B * n <= _SLOPES_KEPT_BYTES:
            trace.slopes[rows.relu] = out
        return out

    def window_conv(rows, p):
        """Window rows through a conv: the pending relu relaxed at their
        places in the image, then the conv of the windows alone; None where
        the window is no longer worth it, or where the relu has an alpha or a
        beta (which gives every neuron of the image a value)."""
        w = rows.window
        C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
        oh, ow = (w.wh - 1) * sh + kh, (w.ww - 1) * sw + kw
        if (not w.worth() or trace is not None or rows.alpha is not None
                or rows.beta is not None
                or (rows.shared and rows.relu is None and not acc_shared)
                or B * R * C_in * oh * ow >= 1 << 31):
            return None
        ls = us = ut = None
        if rows.relu is not None:
            ls, us, ut = slopes(rows)
            bias, acc_b = p['b'], acc
        else:
            bias, acc_b = bias_acc(rows, p)
        M = R if rows.shared and rows.relu is None else B * R
        rel = torch.empty(M, C_out * w.wh * w.ww, device=dev)
        call('vc_patch_relax', ptr(rows.ew), M, R, 1 if rows.shared else 0, ptr(ls), ptr(us),
             ptr(ut), ptr(w.origin), C_out, w.H, w.W, w.wh, w.ww, ptr(rel), ptr(acc), st)
        out = _Rows(torch.empty(M, C_in * oh * ow, device=dev), M == R and rows.shared
                    and rows.relu is None)
        conv_fp32(p, rel, M, (w.wh, w.ww, oh, ow), out.ew, bias, acc_b)
        origin = torch.empty_like(w.origin)
        call('vc_patch_shift', ptr(w.origin), R, sh, sw, ph, pw, ptr(origin), st)
        out.window = _Window(origin, oh, ow, C_in, H, W)
        return out

    def relu_conv(rows, op, p):
        """The pending relu relaxation fused into the conv backward that
        follows it (vc_backward_relu_conv for a few input channels, else
        vc_backward_conv_split), or None when the geometry or the
        relaxation's form is outside the fused kernels."""
        if rows.alpha_group is not None or (rows.alpha is not None and rows.alpha_row):
            return None
        fold = _few_channels(p)
        parts = (None if fold or not split
                 else packs.conv_split(p, B * R, R, rows.shared, st))
        if not fold and parts is None:
            return None
        ls, us, ut = slopes(rows)
        C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
        out = torch.empty(B * R, p['n_in'], device=dev)
        if parts is not None:
            call('vc_backward_conv_split', ptr(rows.ew), B * R, R, 1 if rows.shared else 0,
                 ptr(ls), ptr(us), ptr(ut), ptr(rows.beta), ptr(p['K']), ptr(parts), ptr(p['b']),
                 C_out, Ho, Wo, C_in, H, W, kh, kw, sh, sw, ph, pw, ptr(out), ptr(acc), st)
            return out
        call('vc_backward_relu_conv', ptr(rows.ew), B * R, R, 1 if rows.shared else 0, ptr(ls),
             ptr(us), ptr(ut), ptr(rows.beta), ptr(p['K']), ptr(p['b']), C_out, Ho, Wo, C_in,
             H, W, kh, kw, sh, sw, ph, pw, ptr(out), ptr(acc), st)
        return out

    for op in reversed(ops):
        name = op['name']
        if name not in ew_at:
            continue
        rows = ew_at.pop(name)
        t = op['type']
        inp = op['inputs'][0]
        if rows.window is not None and t not in ('conv', 'relu'):
            rows = dense(rows)
        if t in ('add', 'sub', 'mul') and trace is not None:
            trace.other = trace.other or t
        if t == 'add' and op.get('is_merge'):
            # the rows flow to both branches unchanged (verify_zono_bnb.py:4462-4469)
            rows = materialize(rows)
            for i in op['inputs']:
                put(i, _Rows(rows.ew, rows.shared))
        elif t in ('add', 'sub'):
            # constant shift: acc +/-= rows . bias, rows unchanged
            # (verify_zono_bnb.py:4470-4518)
            rows = materialize(rows)
            b = _op_const(op, 'bias', dev, rows.ew.shape[1])
            if b is not None:
                bias_dot(rows, b, 1.0 if t == 'add' else -1.0)
            put(inp, rows)
        elif t == 'mul':
            # constant scale: rows * scale (verify_zono_bnb.py:4686-4712)
            rows = materialize(rows)
            s = _op_const(op, 'scale', dev, rows.ew.shape[1])
            if s is None:
                raise ValueError(f'mul {name!r}: no scale')
            out = torch.empty_like(rows.ew)
            call('vc_affine_ew', ptr(rows.ew), rows.ew.shape[0], rows.ew.shape[1], 1, ptr(s),
                 s.numel(), 2, ptr(out), st)
            put(inp, _Rows(out, rows.shared))
        elif t == 'fc' and _fc_form(op, widths[inp])[0] > 1:
            # N-D batched MatMul (verify_zono_bnb.py:4382-4401): acc += the
            # rows . bias repeated over the P slices, then each row's P
            # slices of n_out times W, as (M * P, n_out) rows
            P, nd_out = _fc_form(op, widths[inp])
            if not nd_out:
                raise NotImplementedError(
                    f'batched spec backward: fc {name!r} is an N-D batched MatMul '
                    f'without out_shape_nd')
            if trace is not None:
                trace.other = trace.other or 'N-D fc'
            p = _op_params(op, dev)
            rows = materialize(rows)
            if p['b'] is not None:
                bias_dot(rows, p['b'].repeat(P), 1.0)
            M = rows.ew.shape[0]
            out = torch.empty(M, P * p['n_in'], device=dev)
            call('vc_backward_fc', ptr(rows.ew), M * P, R * P, p['n_out'], None,
                 None, None, 0, None, ptr(p['W']), None, p['n_in'], ptr(out), None,
                 None, 0, st)
            put(inp, _Rows(out, rows.shared))
        elif t == 'fc':
            p = _op_params(op, dev)
            if rows.relu is not None:
                L = rows.relu
                M = B * R
                out = torch.empty(M, p['n_in'], device=dev)
                parts = None
                if (split and M >= _FC_SPLIT_SWEEP_ROWS and rows.alpha_group is None
                        and not rows.alpha_row):
                    parts = _fc_split_parts(packs, p, M, st, once=once,
                                            sweep=trace is not None)
                if parts is not None:
                    ls, us, ut = slopes(rows)
                    if trace is not None:
                        trace.fcs.append(op)

                    def launch(d, m, r, M, R, work):
                        call('vc_backward_fc_split',
                             ptr(_cut(rows.ew, r if rows.shared else m)), M, R,
                             1 if rows.shared else 0, p['n_out'], ptr(_cut(ls, d)),
                             ptr(_cut(us, d)), ptr(_cut(ut, d)), ptr(_cut(rows.beta, d)),
                             ptr(parts), ptr(p['b']), p['n_in'], ptr(_cut(out, m)),
                             ptr(_cut(acc, m)), ptr(work), st)
                    _in_slices(B, R, p['n_out'], dev, launch)
                    put(inp, _Rows(out, False))
                    continue
                lo, hi = f32(tight[L][0]), f32(tight[L][1])
                per_domain_acc()
                if trace is not None:
                    trace.relus.append((L, rows.ew, rows.shared))
                    trace.fcs.append(op)
                # the relaxed rows buffer selects the library's two-phase
                # step (relaxation streamed through HBM, then a plain GEMM)
                rel = (torch.empty(M, p['n_out'], device=dev)
                       if p['n_out'] >= _TWO_PHASE_MIN_WIDTH else None)
                if rows.alpha_group is not None:
                    if rows.beta is not None:
                        raise NotImplementedError(
                            'vibecheck_amd: group-indexed alpha takes no beta')
                    call('vc_backward_fc_grouped', ptr(rows.ew), M, R, p['n_out'],
                         ptr(lo), ptr(hi), ptr(rows.alpha), ptr(rows.alpha_group),
                         rows.n_groups, ptr(p['W']), ptr(p['b']), p['n_in'], ptr(out), ptr(acc),
                         ptr(rel), 1 if rows.shared else 0, st)
                else:
                    call('vc_backward_fc', ptr(rows.ew), M, R, p['n_out'],
                         ptr(lo), ptr(hi), ptr(rows.alpha), rows.alpha_row,
                         ptr(rows.beta), ptr(p['W']), ptr(p['b']), p['n_in'],
                         ptr(out), ptr(acc), ptr(rel), 1 if rows.shared else 0, st)
                del rel
                put(inp, _Rows(out, False))
            else:
                bias, acc_b = bias_acc(rows, p)
                M = R if rows.shared else B * R
                out = torch.empty(M, p['n_in'], device=dev)
                if trace is not None:
                    trace.fcs.append(op)
                call('vc_backward_fc', ptr(rows.ew), M, R, p['n_out'], None,
                     None, None, 0, None, ptr(p['W']), ptr(bias),
                     p['n_in'], ptr(out), ptr(acc_b), None, 0, st)
                put(inp, _Rows(out, rows.shared))
        elif t == 'relu':
            if 'layer_idx' in op:
                if rows.relu is not None:
                    rows = materialize(rows)
                L = op['layer_idx']
                rows.relu = L
                if alpha_at_layer is not None and L in alpha_at_layer:
                    a = alpha_at_layer[L]
                    if isinstance(a, tuple):
                        # (alpha of each group (G, R, n), group of each domain (B,))
                        rows.alpha = f32(a[0]).reshape(-1, a[0].shape[-1])
                        rows.alpha_row = 0
                        rows.alpha_group = a[1]
                        rows.n_groups = int(a[0].shape[0])
                        a = None
                    else:
                        a = f32(a)
                    if a is None:
                        pass
                    elif a.dim() == 3:
                        rows.alpha = a.reshape(B * R, -1)
                        rows.alpha_row = 1
                    else:
                        rows.alpha = a
                        rows.alpha_row = 0
                if relu_split_beta is not None and L in relu_split_beta:
                    rows.beta = f32(relu_split_beta[L])
            put(inp, rows)
        elif t == 'conv':
            p = _op_params(op, dev)
            if rows.window is not None:
                out = window_conv(rows, p)
                if out is not None:
                    put(inp, out)
                    continue
                rows = dense(rows)
            if rows.relu is not None and FUSED_RELU_CONV:
                out = relu_conv(rows, op, p)
                if out is not None:
                    put(inp, _Rows(out, False))
                    continue
            rows = materialize(rows)
            C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = p['geom']
            bias, acc_b = bias_acc(rows, p)
            M = R if rows.shared else B * R
            out = torch.empty(M, p['n_in'], device=dev)
            parts = (None if not split or _few_channels(p)
                     else packs.conv_split(p, M, M, False, st))
            if parts is not None:
                call('vc_backward_conv_split', ptr(rows.ew), M, M, 0, None, None, None, None,
                     ptr(p['K']), ptr(parts), ptr(bias), C_out, Ho, Wo, C_in, H, W, kh, kw,
                     sh, sw, ph, pw, ptr(out), ptr(acc_b), st)
                put(inp, _Rows(out, rows.shared))
                continue
            conv_fp32(p, rows.ew, M, None, out, bias, acc_b)
            put(inp, _Rows(out, rows.shared))
        elif t == 'reshape':
            put(inp, rows)
        else:
            raise ValueError(f'batched spec backward: unknown op {t!r}')

    rows = ew_at.get(gg['input_name'])
    if rows is None:
        per_domain_acc()
        return acc.reshape(B, R).clone(), None, False, acc
    lb = torch.empty(B * R, device=dev)
    if rows.window is not None and rows.relu is None:
        per_domain_acc()
        w = rows.window
        call('vc_patch_concretize', ptr(rows.ew), 1 if rows.shared else 0, ptr(w.origin),
             ptr(acc), ptr(xl), ptr(xh), B * R, R, w.C, w.H, w.W, w.wh, w.ww, ptr(lb), st)
        return lb.reshape(B, R), None, False, acc
    rows = materialize(rows)
    A = rows.ew
    per_domain_acc()
    call('vc_concretize', ptr(A), ptr(acc), ptr(xl), ptr(xh), B * R, R, n_in,
         1 if rows.shared else 0, ptr(lb), st)
    return lb.reshape(B, R), A, rows.shared, acc


_SPEC_CACHE = {}


def _spec_rows(spec_ew, dev):
    """The spec rows stacked (Q, n_out) and their offsets (Q,) on ``dev``.
    Cached for tensor rows (keyed on each tensor's identity and in-place
    version): building them copies the offsets from the host, which would
    stall the stream once per bound call.  Callers only read the result."""
    qids = sorted(spec_ew.keys())
    key = None
    if all(torch.is_tensor(spec_ew[q][0]) and not torch.is_tensor(spec_ew[q][1])
           for q in qids):
        key = (str(dev), tuple((q, id(spec_ew[q][0]), spec_ew[q][0]._version,
                                float(spec_ew[q][1])) for q in qids))
        hit = _SPEC_CACHE.get(key)
        if hit is not None:
            return hit[1], hit[2]
    Wq = torch.stack([torch.as_tensor(spec_ew[q][0]).reshape(-1)
                      .to(device=dev, dtype=torch.float32) for q in qids]).contiguous()
    bq = torch.tensor([float(spec_ew[q][1]) for q in qids],
                      dtype=torch.float32, device=dev)
    if key is not None:
        if len(_SPEC_CACHE) >= 32:
            _SPEC_CACHE.pop(next(iter(_SPEC_CACHE)))
        # the rows are held so that their identities stay unique
        _SPEC_CACHE[key] = ([spec_ew[q][0] for q in qids], Wq, bq)
    return Wq, bq


def _spec_backward_graph_batched(tight, xl, xh, gg, spec_ew, device, dtype,
                                 return_input_linear=False,
                                 alpha_at_layer=None, relu_split_beta=None,
                                 alpha_mccormick=None, alpha_recip=None,
                                 bilinear_op_bounds=None, seed_ew_at=None,
                                 seed_acc=None):
    """Batched CROWN spec backward + concretization
    (verify_zono_bnb.py:4270-5134; fc/relu/conv/reshape ops).

    Returns lb (B, Q), or (lb, A (B, Q, n_in), acc (B, Q)) with
    ``return_input_linear``.
    """
    _check_dtype(dtype)
    if alpha_mccormick or alpha_recip or bilinear_op_bounds:
        raise NotImplementedError(
            'vibecheck_amd: bilinear / reciprocal relaxations are not '
            'supported (Linear/Conv/ReLU networks only)')
    xl, xh = f32(xl), f32(xh)
    _widths(gg, xl.shape[1])
    B, n_in = xl.shape
    dev = xl.device
    plan = _plan(gg, dev)
    if (plan is not None and seed_ew_at is None and alpha_at_layer is None
            and relu_split_beta is None and len(spec_ew) <= 32):
        Wq, bq = _spec_rows(spec_ew, dev)
        sb = {L: (f32(tight[L][0]), f32(tight[L][1])) for L in range(plan.n)}
        _, lb, A, acc = mlp_fused.crown(plan, xl, xh, sb, False, spec=(Wq, bq),
                                        want_linear=return_input_linear)
        return (lb, A, acc) if return_input_linear else lb
    if seed_ew_at is not None:
        if len(seed_ew_at) != 1:
            raise NotImplementedError('vibecheck_amd: one seed node only')
        seed_name, seed = next(iter(seed_ew_at.items()))
        Q = seed.shape[1]
        if seed.dim() == 3 and seed.stride(0) == 0:
            rows, shared = f32(seed[0]).contiguous(), True
        else:
            rows, shared = f32(seed).reshape(B * Q, -1).contiguous(), False
        if seed_acc is None:
            acc0 = torch.zeros(Q if shared else B * Q, device=dev)
        else:
            sa = f32(seed_acc)
            if shared and sa.stride(0) == 0:
                acc0 = sa[0].contiguous().clone()
            else:
                if shared:
                    rows, shared = _expand_rows(rows, B), False
                acc0 = sa.reshape(B * Q).contiguous().clone()
    else:
        rows, acc0 = _spec_rows(spec_ew, dev)
        seed_name, shared = gg['ops'][-1]['name'], True
        Q = rows.shape[0]
    lb, A, a_shared, acc = _backward(tight, xl, xh, gg, seed_name, rows,
                                     shared, acc0, alpha_at_layer,
                                     relu_split_beta)
    if not return_input_linear:
        return lb
    if A is None:
        return lb, torch.zeros(B, Q, n_in, device=dev), acc.reshape(B, Q)
    if a_shared:
        A = A.unsqueeze(0).expand(B, Q, n_in).contiguous()
    else:
        A = A.reshape(B, Q, n_in)
    return lb, A, acc.reshape(B, Q)


# --------------------------------------------------------------------------
# a4: CROWN intermediate bounds
# --------------------------------------------------------------------------

def _crown_intermediate_batched(gg, xl, xh, device, dtype, chunk=2048,
                                sb=None):
    """Backward-CROWN intermediate pre-ReLU bounds
    (verify_zono_bnb.py:4077-4147).

    For each ReLU layer L in ascending order: seed [+I; -I] at L's input for
    the neurons unstable in ANY domain of the batch, in chunks of ``chunk``,
    propagate through the already-tightened earlier layers and intersect.
    The seeded rows are identical for every domain until the first ReLU, so
    that prefix is computed once (R rows) and broadcast.  ``sb`` (extension)
    replaces the zonotope starting bounds, e.g. by IBP bounds.
    """
    _check_dtype(dtype)
    xl, xh = f32(xl), f32(xh)
    _widths(gg, xl.shape[1])
    dev = xl.device
    if sb is None:
        sb = _zono_sb(gg, xl, xh, device, dtype)
    plan = _plan(gg, dev)
    if plan is not None:
        tight, _, _, _ = mlp_fused.crown(
            plan, xl, xh, {L: (f32(sb[L][0]), f32(sb[L][1])) for L in range(plan.n)}, True)
        return tight
    tight = {L: (f32(lo).clone(), f32(hi).clone()) for L, (lo, hi) in sb.items()}
    relu_by_L = {op['layer_idx']: op for op in gg['ops']
                 if op['type'] == 'relu' and 'layer_idx' in op}
    B = xl.shape[0]
    st = stream()
    packs = _Packs(gg, dev)
    ch = max(1, int(chunk))
    for L in sorted(tight):
        if L not in relu_by_L:
            continue
        feed = relu_by_L[L]['inputs'][0]
        lo_L, hi_L = tight[L]
        n = lo_L.shape[1]
        flag = torch.empty(n, dtype=torch.uint8, device=dev)
        call('vc_unstable_union', ptr(lo_L), ptr(hi_L), B, n, ptr(flag), st)
        idx = flag.nonzero(as_tuple=True)[0].to(torch.int32)
        m = int(idx.numel())
        if m == 0:
            continue
        new_lo, new_hi = lo_L.clone(), hi_L.clone()
        window = below = None
        feed_op = next(op for op in gg['ops'] if op['name'] == feed)
        if feed_op['type'] == 'conv':
            p = _op_params(feed_op, dev)
            C_in, H, W, _, kh, kw = p['geom'][:6]
            if p['n_out'] <= 1 << 30 and _Window(None, kh, kw, C_in, H, W).worth():
                window, below = p, feed_op['inputs'][0]
        for c0 in range(0, m, ch):
            cidx = idx[c0:c0 + ch].contiguous()
            k = int(cidx.numel())
            if window is not None:
                # one conv neuron's row is its own kernel, a window of the
                # conv's input (and acc its bias): no product, no whole rows
                C_in, H, W, C_out, kh, kw, sh, sw, ph, pw, Ho, Wo = window['geom']
                rows = _Rows(torch.empty(2 * k, C_in * kh * kw, device=dev), True)
                origin = torch.empty(2 * k, 2, dtype=torch.int32, device=dev)
                acc0 = torch.empty(2 * k, device=dev)
                call('vc_patch_seed', ptr(window['K']), ptr(window['b']), ptr(cidx), k, C_out,
                     Ho, Wo, C_in, kh, kw, sh, sw, ph, pw, ptr(rows.ew), ptr(origin), ptr(acc0),
                     st)
                rows.window = _Window(origin, kh, kw, C_in, H, W)
                sl, _, _, _ = _backward(tight, xl, xh, gg, below, rows, True, acc0,
                                        split=False, packs=packs, fresh=True)
                call('vc_crown_intersect', ptr(sl.contiguous()), ptr(cidx), k, B, n,
                     ptr(new_lo), ptr(new_hi), st)
                continue
            seed = torch.zeros(2 * k, n, device=dev)
            ar = torch.arange(k, device=dev)
            seed[ar, cidx.long()] = 1.0
            seed[ar + k, cidx.long()] = -1.0
            acc0 = torch.zeros(2 * k, device=dev)
            sl, _, _, _ = _backward(tight, xl, xh, gg, feed, seed, True, acc0, split=False,
                                    packs=packs, fresh=True)
            sl = sl.contiguous()
            call('vc_crown_intersect', ptr(sl), ptr(cidx), k, B, n,
                 ptr(new_lo), ptr(new_hi), st)
        tight[L] = (new_lo, new_hi)
    return tight


# --------------------------------------------------------------------------
# a9: alpha-CROWN
# --------------------------------------------------------------------------

def _alpha_backward_and_grad(sb, xl, xh, gg, Wq, bq, alpha, want_grad, galpha,
                             beta=None, gbeta=None, seed_name=None, want_A=False, packs=None):
    """One alpha-CROWN evaluation: lb (B, Q); when ``want_grad`` also fills
    ``galpha[L]`` with d(sum lb)/d alpha_L (the autograd of the reference's
    backward, torch clamp subgradients included).  ``beta`` is the signed
    ReLU-split beta {L: (B, n_L)} added at each relu's input
    (``relu_split_beta``); ``gbeta[L]`` receives d(sum lb)/d beta_L.
    ``seed_name`` (default: the output op) is the op whose output the Q
    shared rows Wq (Q, n) seed, as ``seed_ew_at`` does; an alpha_L of shape
    (B, Q, n_L) is one alpha per row (per-query alpha), and galpha_L then
    has that shape too.  ``want_A``: returns (lb, A) with A (B*Q, n_in) the
    input linearization of the rows.  ``packs``: the loop's _Packs."""
    B, n_in = xl.shape
    Q = Wq.shape[0]
    dev = xl.device
    packs = _Packs(gg, dev) if packs is None else packs
    st = stream()
    trace = BackwardTrace() if want_grad else None
    seed = gg['ops'][-1]['name'] if seed_name is None else seed_name
    lb, A, a_shared, _ = _backward(sb, xl, xh, gg, seed, Wq,
                                   True, bq, alpha, beta, trace, packs=packs)
    if want_A and (A is None or a_shared):
        raise NotImplementedError('vibecheck_amd: per-row linearization needs a relu')
    if not want_grad:
        return (lb, A) if want_A else lb
    if A is None or a_shared:
        raise NotImplementedError('vibecheck_amd: alpha gradient needs a relu')
    if trace.other is not None:
        raise NotImplementedError(
            f'vibecheck_amd: alpha-CROWN gradient supports fc/relu chains (found {trace.other})')
    # trace.relus: (L, P, shared) in backward order (top relu first);
    # trace.fcs: fc ops in backward order.  Sequential fc/relu nets only:
    # fcs[i] sits below relus[i-1] ... check the chain shape.
    relus = trace.relus
    fcs = trace.fcs
    if len(fcs) != len(relus) + 1:
        raise NotImplementedError(
            'vibecheck_amd: alpha-CROWN gradient supports fc/relu chains')
    M = B * Q
    # input side: gE_0 = gA W_0^T + b_0, W_0 = fcs[-1]
    f0 = _op_params(fcs[-1], dev)
    g = torch.empty(M, f0['n_out'], device=dev)
    parts = _fc_split_parts(packs, f0, M, st, True)
    if parts is not None:
        _in_slices(B, Q, n_in, dev, lambda d, m, r, M, Q, work: call(
            'vc_alpha_grad_input_split', ptr(_cut(A, m)), ptr(_cut(xl, d)), ptr(_cut(xh, d)), M,
            Q, n_in, ptr(parts), ptr(f0['b']), f0['n_out'], ptr(_cut(g, m)), ptr(work), st))
    else:
        call('vc_alpha_grad_input', ptr(A), ptr(xl), ptr(xh), M, Q, n_in,
             ptr(f0['W']), ptr(f0['b']), f0['n_out'], ptr(g), st)
    for i in range(len(relus) - 1, -1, -1):
        L, P, p_shared = relus[i]
        lo, hi = f32(sb[L][0]), f32(sb[L][1])
        n = lo.shape[1]
        a = f32(alpha[L]) if (alpha is not None and L in alpha) else None
        per_row = a is not None and a.dim() == 3
        ga = galpha.get(L) if galpha is not None else None
        gb = gbeta.get(L) if gbeta is not None else None
        if per_row and ga is not None:
            if i == 0:  # above the input: no gradient step to fuse it into
                call('vc_alpha_grad_rows', ptr(g), ptr(P), 1 if p_shared else 0, M, Q, n,
                     ptr(lo), ptr(hi), ptr(ga), st)
            ga_rows = ga
            ga = None
        else:
            ga_rows = None
        if ga is not None or gb is not None:
            call('vc_alpha_grad_reduce', ptr(g), ptr(P), 1 if p_shared else 0,
                 B, Q, n, ptr(lo), ptr(hi), ptr(ga), ptr(gb), st)
        if i > 0 and per_row:
            fn = _op_params(fcs[i], dev)
            g2 = torch.empty(M, fn['n_out'], device=dev)
            call('vc_alpha_grad_step_rows', ptr(g), ptr(P), M, Q, n, ptr(lo), ptr(hi),
                 ptr(a.reshape(M, n)), 1 if p_shared else 0, ptr(fn['W']), ptr(fn['b']),
                 fn['n_out'], ptr(g2), ptr(ga_rows), st)
            g = g2
        elif i > 0:
            fn = _op_params(fcs[i], dev)
            g2 = torch.empty(M, fn['n_out'], device=dev)
            # slopes once per (domain, neuron), then the sweep step without
            # a per-element division
            if L in trace.slopes:
                ls, us, ut = trace.slopes[L]
            else:
                ls, us, ut = (torch.empty(B, n, device=dev) for _ in range(3))
                call('vc_relax_slopes', ptr(lo), ptr(hi), ptr(a), B * n, ptr(ls),
                     ptr(us), ptr(ut), st)
            parts = _fc_split_parts(packs, fn, M, st, True)
            if parts is not None:
                _in_slices(B, Q, n, dev, lambda d, m, r, M, Q, work: call(
                    'vc_alpha_grad_step_split', ptr(_cut(g, m)),
                    ptr(_cut(P, r if p_shared else m)), M, Q, n, ptr(_cut(ls, d)),
                    ptr(_cut(us, d)), ptr(_cut(ut, d)), 1 if p_shared else 0, ptr(parts),
                    ptr(fn['b']), fn['n_out'], ptr(_cut(g2, m)), ptr(work), st))
            else:
                call('vc_alpha_grad_step_slopes', ptr(g), ptr(P), M, Q, n,
                     ptr(ls), ptr(us), ptr(ut), 1 if p_shared else 0,
                     ptr(fn['W']), ptr(fn['b']), fn['n_out'], ptr(g2), st)
            g = g2
    return (lb, A) if want_A else lb


def _run_alpha_crown_inputsplit_batched(xl, xh, gg, spec_ew, device, dtype,
                                        n_iters=10, lr=0.25, lr_decay=0.98,
                                        early_stop_eps=1e-6, sb=None,
                                        return_trace=False, lazy_trace=False):
    """Batched alpha-CROWN with Adam (verify_zono_bnb.py:5137-5288).

    Same schedule as the reference: alpha starts at (up_s > 0.5)*unstable on
    the zonotope bounds; per iteration: evaluate, keep the best lb, stop if
    every best lb > 0, Adam step (torch.optim.Adam defaults) on -sum(lb),
    clamp alpha to [0, 1], stop if the global max of the best lb improved by
    less than ``early_stop_eps`` (from the second iteration), decay lr.
    The gradient is computed analytically by the HIP gradient sweep.
    ``sb`` (extension) replaces the zonotope bounds; ``return_trace`` also
    returns the number of evaluated iterations; with ``lazy_trace`` that
    number may come as a callable, to be called after a later host
    synchronisation (it then costs no round trip of its own).
    """
    _check_dtype(dtype)
    xl, xh = f32(xl), f32(xh)
    _widths(gg, xl.shape[1])
    B = xl.shape[0]
    dev = xl.device
    st = stream()
    if sb is None:
        sb = _zono_sb(gg, xl, xh, device, dtype)
    sb = {L: (f32(lo), f32(hi)) for L, (lo, hi) in sb.items()}
    if n_iters < 1 and sb:
        # every ReLU layer is an Adam parameter, the loop body never runs:
        # no best bound (verify_zono_bnb.py:5169-5173, 5247-5288)
        return (None, 0) if return_trace else None
    Wq, bq = _spec_rows(spec_ew, dev)
    Q = Wq.shape[0]
    plan = _plan(gg, dev)
    if plan is not None and mlp_fused.alpha_supported(plan, Q):
        best, n_eval = mlp_fused.alpha_crown(plan, xl, xh, sb, Wq, bq, n_iters, lr,
                                             lr_decay, early_stop_eps, lazy=lazy_trace)
        return (best, n_eval) if return_trace else best
    Ls = sorted(sb)
    sizes = [sb[L][0].numel() for L in Ls]
    total = sum(sizes)
    if total == 0:
        lb = _alpha_backward_and_grad(sb, xl, xh, gg, Wq, bq, None, False,
                                      None)
        return (lb, 1) if return_trace else lb
    flat = torch.empty(total, device=dev)
    gflat = torch.zeros(total, device=dev)
    m1 = torch.zeros(total, device=dev)
    m2 = torch.zeros(total, device=dev)
    alpha, galpha = {}, {}
    off = 0
    for L, sz in zip(Ls, sizes):
        alpha[L] = flat[off:off + sz].view(sb[L][0].shape)
        galpha[L] = gflat[off:off + sz].view(sb[L][0].shape)
        call('vc_alpha_init', ptr(sb[L][0]), ptr(sb[L][1]), sz,
             ptr(alpha[L]), st)
        off += sz
    best = torch.empty(B, Q, device=dev)
    red = torch.empty(2, device=dev)
    b1, b2, eps = 0.9, 0.999, 1e-8
    prev_max = -float('inf')
    n_eval = 0
    step = 0
    cur_lr = float(lr)
    packs = _Packs(gg, dev)
    for it in range(n_iters):
        lb = _alpha_backward_and_grad(sb, xl, xh, gg, Wq, bq, alpha, True,
                                      galpha, packs=packs)
        n_eval += 1
        call('vc_best_update', ptr(best), ptr(lb.contiguous()), B * Q,
             1 if it == 0 else 0, ptr(red), st)
        r = red.tolist()
        curr_max, all_pos = r[0], r[1] > 0.5
        if all_pos:
            break
        step += 1
        bc1 = 1 - b1 ** step
        bc2 = 1 - b2 ** step
        call('vc_adam_step', ptr(flat), ptr(gflat), ptr(m1), ptr(m2), total,
             b1, b2, eps, cur_lr / bc1, bc2 ** 0.5, 0.0, 1.0, st)
        if it > 0 and curr_max - prev_max < early_stop_eps:
            break
        prev_max = curr_max
        cur_lr *= lr_decay
    if return_trace:
        return best, n_eval
    return best


def _bound_crown_spec(gg, xl, xh, spec_ew, device, dtype,
                      return_input_linear=False, return_zono_sb=False, union_seeds=False):
    """CROWN intermediate bounds followed by the spec bound -- the 'bound'
    phase of an input-split BaB iteration (verify_graph.py:12855-12871).
    For narrow fc/ReLU chains both run in one whole-network kernel launch,
    which by default seeds in each domain only the union neurons whose
    slopes depend on their bounds there: the spec bound, A and acc are
    those of the reference's union seeding, and so are the bounds of every
    neuron unstable in the domain; the bounds of the domain's stable
    neurons stay the zonotope ones (``union_seeds=True`` tightens them
    too, as _crown_intermediate_batched does).
    Returns (tight, lb) or (tight, lb, A, acc); ``return_zono_sb``
    (extension) appends the zonotope bounds the CROWN pass started from,
    which the alpha-CROWN of the same boxes starts from as well."""
    _check_dtype(dtype)
    xl, xh = f32(xl), f32(xh)
    plan = _plan(gg, xl.device)
    sb = _zono_sb(gg, xl, xh, device, dtype)
    if plan is not None and len(spec_ew) <= 32:
        Wq, bq = _spec_rows(spec_ew, xl.device)
        tight, lb, A, acc = mlp_fused.crown(plan, xl, xh, sb, True, spec=(Wq, bq),
                                            want_linear=return_input_linear,
                                            per_domain=not union_seeds)
        out = (tight, lb, A, acc) if return_input_linear else (tight, lb)
    else:
        tight = _crown_intermediate_batched(gg, xl, xh, device, dtype, sb=sb)
        res = _spec_backward_graph_batched(tight, xl, xh, gg, spec_ew, device, dtype,
                                           return_input_linear=return_input_linear)
        out = (tight,) + tuple(res) if return_input_linear else (tight, res)
    return out + (sb,) if return_zono_sb else out
