"""Workloads of the dedispersion chain and of the learned scorer, for timing and for comparing
two builds of the library.

A case is a dict of plain values. Kinds:

  chain  one chunk of every beam through a GpuDedisperser, as a search program runs it: packed
         int4 samples (on the GPU, as they arrive from the network) are dequantized into the
         acquired input slot, the chain is launched and its outputs are acquired.
  group  the same for a GpuDedisperserGroup: beam groups of several tree ranks, one chunk of all.
  score  LearnedScorer.forward on a batch of (DM, time) tiles.
  train  LearnedScorer.train_step on a batch of labelled tiles.

Chain cases carry the fields of a dedispersion config: nfreq and edges (frequency zones), rank
(toplevel tree rank), chunk (samples), beams, batch (beams per batch), active (batches in
flight), bands (frequency subband counts), widths and triggers (largest boxcar and early triggers
of each primary tree), dtype, and scorer (the learned scorer inside the chain).

listed() gives the fixed cases, draw() more of the same ranges, prepare() the state a program
keeps, run() one pass, work() the bytes and operations a pass cannot do without, exact() the
outputs in float64 by plain torch.
"""

import math

import numpy as np
import torch

import pirate_amd as pa

NCHUNK = 3                    # resident chunks: two go through the chain before the first pass
SIZE = {'float32': 4, 'float16': 2, 'bfloat16': 2}
ROWS, COLS, TAPS, CH = 64, 256, 9, 16      # scorer tile and network


def chain(name, **kw):
    d = dict(name=name, kind='chain', dtype='float32', nfreq='1024', edges='400,800', rank=10, chunk=2048, beams=1,
             batch=1, active=1, bands='1', widths='16', triggers='0', scorer=False)
    d.update(kw)
    return d


def listed():
    return [
        # The smallest search: a toy-sized config with early triggers and a subband search, its
        # two batches in flight together. Launches and host work dominate.
        chain('toy', nfreq='640', rank=8, chunk=256, beams=4, batch=2, active=2, bands='2,2,1', widths='16,8,4',
              triggers='0,1,1'),
        # One beam of a small telescope: latency of a chunk.
        chain('one_beam'),
        # Irregular zones, an odd beam count, a chunk whose coarsest tree ends in half a tile.
        chain('ragged', nfreq='201,299,503', edges='300,500,800,1500', rank=11, chunk=768, beams=5,
              batch=5, bands='3,3,1', widths='8,4,4,2', triggers='1,0,0,1'),
        # The scorer's own training chain: 16 beams of 1024 channels, scored in the chain.
        chain('scored_16_beams', beams=16, batch=16, scorer=True),
        # A wide subband search over two primary trees, boxcars up to 32 samples, bfloat16 storage.
        chain('subbands_r12_bf16', dtype='bfloat16', nfreq='4096', edges='300,1500', rank=12, beams=8, batch=8, bands='4,5,3,1', widths='32,16'),
        # The headline: 16 beams x 16384 channels, four primary trees; and its 16-bit storage.
        chain('chord16k_f32', nfreq='16384', edges='300,1500', rank=14, beams=16, batch=16, widths='16,8,4,2',
              triggers='0,0,0,0'),
        chain('chord16k_f16', dtype='float16', nfreq='16384', edges='300,1500', rank=14, beams=16, batch=16,
              widths='16,8,4,2', triggers='0,0,0,0'),
        # Production shapes: rank 15 with a subband search, rank 16 full band.
        chain('rank15_subbands_f16', dtype='float16', nfreq='16384', rank=15, beams=8, batch=8, bands='0,0,1,2,1',
              widths='16,8,4,2', triggers='0,0,0,0'),
        chain('rank16_f16', dtype='float16', nfreq='28160', edges='300,1500', rank=16, beams=4, batch=4, bands='0,0,0,0,1',
              widths='16,8,4,2', triggers='0,0,0,0'),
        # 96 beams of three shapes as one group.
        dict(name='group_96_beams', kind='group', dtype='float16', ranks='12,13,14', beams=32, chunk=2048),
        # Scoring a chunk's candidates, and one training step at the trainer's batch size.
        dict(name='score_8192', kind='score', dtype='bfloat16', tiles=8192),
        dict(name='train_512', kind='train', dtype='bfloat16', tiles=512),
    ]


def draw(rng):
    kind = rng.choice(['chain'] * 6 + ['group', 'score', 'train'])
    if kind in ('score', 'train'):
        hi = 16384 if kind == 'score' else 4096
        return dict(kind=kind, dtype=rng.choice(['float32', 'float16', 'bfloat16']),
                    tiles=int(round(math.exp(rng.uniform(math.log(3), math.log(hi))))))
    if kind == 'group':
        ranks = sorted(rng.sample([10, 11, 12, 13, 14], rng.choice([2, 3])))
        return dict(kind='group', dtype=rng.choice(['float32', 'float16', 'bfloat16']), ranks=','.join(map(str, ranks)),
                    beams=rng.randint(1, 12), chunk=rng.choice([1024, 1536, 2048]))
    while True:
        dtype = rng.choice(['float32', 'float16', 'bfloat16'])
        rank = rng.randint(8, 16)
        npri = rng.randint(1, 5)
        chunk = 256 * rng.randint(1, 12)
        if chunk % ((128 // SIZE[dtype]) << (npri - 1)) or (npri > 1 and (chunk >> (npri - 1)) < 1 << ((rank - 1) // 2)):
            continue
        active = rng.choice([1, 1, 2])
        batch = rng.randint(1, 16)
        beams = batch * active
        bands = rng.choice(['1', '1', '2,1', '2,2,1', '0,3,1', '4,5,3,1', '0,0,0,0,1', '0,0,1,2,1'])
        most = 16 if sum(ints(bands)) == 1 else 8          # chunks of 2048 samples at rank 14
        if beams * (chunk << rank) > most * (2048 << 14):
            continue
        nfreq = int(round(math.exp(rng.uniform(math.log(2 ** (rank - 2)), math.log(1.5 * 2 ** rank)))))
        edges = rng.choice(['400,800', '300,1500', '300,600,1500'])
        if edges.count(',') == 2:
            n1 = int(nfreq * rng.uniform(0.3, 0.7))
            nfreq = '%d,%d' % (n1, nfreq - n1)
        triggers = [rng.choice([0, 0, 0, 1]) if rank >= 9 else 0 for _ in range(npri)]
        widths = [rng.choice([32, 16, 8]) if p == 0 else rng.choice([16, 8, 4, 2, 1]) for p in range(npri)]
        return dict(kind='chain', dtype=dtype, nfreq=str(nfreq), edges=edges,
                    rank=rank, chunk=chunk, beams=beams, batch=batch, active=active, bands=bands,
                    widths=','.join(map(str, widths)), triggers=','.join(map(str, triggers)), scorer=False)


# ---------------------------------------------------------------------------------------------
# Configs and tree shapes

def ints(text):
    return [int(x) for x in str(text).split(',')]


def chains_of(case):
    """The chain cases a case is made of: itself, or a group's members."""
    if case['kind'] == 'chain':
        return [case]
    out = []
    for r in ints(case['ranks']):
        npri = max(1, r - 9)
        while case['chunk'] % ((128 // SIZE[case['dtype']]) << (npri - 1)) or (npri > 1 and (case['chunk'] >> (npri - 1)) < 1 << ((r - 1) // 2)):
            npri -= 1
        out.append(chain('member', dtype=case['dtype'], nfreq=str(1 << r), edges='300,1500', rank=r, chunk=case['chunk'],
                         beams=case['beams'], batch=case['beams'], widths=','.join(['16', '8', '4', '2', '1'][:npri]),
                         triggers=','.join(['0'] * npri)))
    return out


def wt_time(nt):
    """Weight time resolution of a tree of nt samples: 64 samples, or the largest power of two that divides nt."""
    return min(64, nt & -nt)


def config(case):
    pts = [dict(num_early_triggers=e, max_width=w, dm_downsampling=0, time_downsampling=0, wt_dm_downsampling=64,
                wt_time_downsampling=wt_time(case['chunk'] >> p))
           for p, (e, w) in enumerate(zip(ints(case['triggers']), ints(case['widths'])))]
    return dict(zone_nfreq=ints(case['nfreq']), zone_freq_edges=ints(case['edges']), toplevel_tree_rank=case['rank'],
                time_samples_per_chunk=case['chunk'], time_sample_ms=1.0, dtype=case['dtype'],
                beams_per_gpu=case['beams'], beams_per_batch=case['batch'], num_active_batches=case['active'],
                frequency_subband_counts=ints(case['bands']), primary_trees=pts, future_write_max_samples=0)


def restricted(counts, et, new_rank):
    """Subband counts of an early-trigger tree whose peak finder resolves 2^new_rank bands."""
    top = max(len(counts) - 1 - et, 0)
    cut = [min(counts[lev], 2 ** (top + 1 - lev) - 1 if lev else 2 ** top) for lev in range(top)] + [1]
    out = []
    for lev in range(new_rank):
        s = lev - new_rank + top
        if s < 0 or cut[s] == 0:
            out.append(0)
        elif s == 0 and lev > 0:
            out.append(2 * cut[0] - 1)
        elif s > 0 and lev == 0:
            out.append(cut[s] // 2 + 1)
        else:
            out.append(cut[s])
    return out + [1]


def trees(case):
    """Output trees in order: primary tree p, channels' rank rr, subband counts, shapes."""
    out = []
    R = case['rank']
    for p, (ets, width) in enumerate(zip(ints(case['triggers']), ints(case['widths']))):
        prank = R - 1 if p else R
        for et in range(ets, -1, -1):
            dd = prank - prank // 2 - et
            pf = (dd + 1) // 2
            nt = case['chunk'] >> p
            tot = prank - et
            counts = restricted(ints(case['bands']), et, pf)
            P = 1 + 3 * (width.bit_length() - 1)
            out.append(dict(p=p, rr=R - et, tot=tot, pf=pf, counts=counts, N=sum(counts),
                            M=sum(c << lev for lev, c in enumerate(counts)), nt=nt, width=width, P=P, dout=1 << pf,
                            ndm=1 << (tot - pf), nt_out=nt >> pf, ndm_wt=1 << (tot - 6), nt_wt=nt // wt_time(nt)))
    return out


# ---------------------------------------------------------------------------------------------
# Inputs

def device():
    return 'cuda' if torch.cuda.is_available() else 'cpu'


def generator(*key):
    g = torch.Generator(device=device())
    g.manual_seed(int(np.random.SeedSequence([int(k) for k in key]).generate_state(1, np.uint64)[0] >> np.uint64(1)))
    return g


def channel_edges(case):
    """Channel edges in MHz, from the lowest."""
    n, e = ints(case['nfreq']), ints(case['edges'])
    return np.concatenate([np.linspace(e[i], e[i + 1], n[i], endpoint=False) for i in range(len(n))] + [[e[-1]]])


def packed_chunk(case, beams, seed, ichunk):
    """One chunk of int4 samples and their float16 scales and offsets: unit-variance noise, one
    dispersed pulse per beam, and blocks of missing samples (value -8)."""
    F, T = sum(ints(case['nfreq'])), case['chunk']
    f = channel_edges(case)[:-1]
    delay = (f ** -2.0 - f[-1] ** -2.0) / (f[0] ** -2.0 - f[-1] ** -2.0)
    delay = torch.from_numpy(delay).to(device())
    ff = torch.arange(F, device=device())
    data = torch.empty((beams, F, T // 2), dtype=torch.uint8, device=device())
    rng = np.random.default_rng([seed, ichunk, 17])
    g = generator(seed, ichunk, 1)
    step = 0.35
    for b in range(beams):
        x = torch.randn((F, T), generator=g, device=device())
        width = int(2 ** rng.uniform(0, 4))
        shift = (delay * float(rng.uniform(1, T / 2)) + float(rng.uniform(0, T))).long()
        for w in range(width):
            x[ff, (shift + w) % T] += 20.0 / math.sqrt(F * width)
        q = torch.clamp(torch.round(x / step), -7, 7).to(torch.int16)
        lost = torch.rand((F, T // 256, 1), generator=g, device=device()) < 0.005
        q = torch.where(lost, torch.full_like(q.view(F, T // 256, 256), -8), q.view(F, T // 256, 256)).view(F, T) & 15
        data[b] = (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8)
    scoff = torch.empty((beams, F, T // 256, 2), dtype=torch.float16, device=device())
    scoff[..., 0] = step * (0.9 + 0.2 * torch.rand(scoff.shape[:3], generator=g, device=device()))
    scoff[..., 1] = 0.05 * torch.randn(scoff.shape[:3], generator=g, device=device())
    return data, scoff


def weight_factors(t, seed, itree):
    """float32 (ndm_wt, nt_wt) factors of a tree's weights, and (P,) bare profile weights."""
    rng = np.random.default_rng([seed, itree, 29])
    f = rng.uniform(0.7, 1.0, size=(t['ndm_wt'], t['nt_wt'])).astype(np.float32)
    var = [1.0] + [2.0 ** lev * v for lev in range((t['P'] - 1) // 3) for v in (2.0, 1.5, 2.5)]
    return f, (1.0 / np.sqrt(np.array(var))).astype(np.float32)


def network(seed):
    """Parameters of the scorer, in its order, float64."""
    rng = np.random.default_rng([seed, 41])
    parts = [rng.standard_normal(CH * ROWS * TAPS) * math.sqrt(2.0 / (ROWS * TAPS)),
             rng.standard_normal(2 * CH * CH * TAPS) * math.sqrt(2.0 / (CH * TAPS)),
             rng.standard_normal(3 * CH) * 0.1, rng.standard_normal(2 * CH) * 0.25, np.zeros(1)]
    return np.concatenate(parts).astype(np.float32).astype(np.float64)


def tile_batch(case, seed):
    """(n, 64, 256) tiles of noise, half of them with a pulse around the centre, and labels."""
    n = case['tiles']
    g = generator(seed, 3)
    x = torch.randn((n, ROWS, COLS), generator=g, device=device())
    y = (torch.rand(n, generator=g, device=device()) < 0.5).to(torch.float32)
    amp = 1.0 + 2.0 * torch.rand((n, 1, 1), generator=g, device=device())
    slope = 2.0 * torch.rand((n, 1, 1), generator=g, device=device()) - 1.0
    r = torch.arange(ROWS, device=device()).view(1, -1, 1) - ROWS / 2
    c = torch.arange(COLS, device=device()).view(1, 1, -1) - COLS / 2
    x += y.view(-1, 1, 1) * amp * torch.exp(-((c - slope * r) / 6.0) ** 2 - (r / 20.0) ** 2)
    return x.to(getattr(torch, case['dtype'])), y


# ---------------------------------------------------------------------------------------------
# State and pass

class ChainState:
    def __init__(self, case, seed):
        self.dd = pa.GpuDedisperser(pa.DedispersionPlan(pa.DedispersionConfig.from_dict(config(case))))
        self.dd.allocate()
        fill_weights(self.dd, case, seed)
        if case['scorer']:
            self.dd.set_scorer(network(seed), 0)
        B, F, T = case['batch'], self.dd.nfreq, case['chunk']
        self.dequantize = pa.GpuDequantizationKernel(case['dtype'], B, F, T)
        self.scored = case['scorer']
        whole = [packed_chunk(case, case['beams'], seed, c) for c in range(NCHUNK)]
        self.chunks = [[(d[i:i + B], s[i:i + B]) for i in range(0, case['beams'], B)] for d, s in whole]
        self.seq = 0
        for _ in range(NCHUNK - 1):
            self.one_chunk()

    def one_chunk(self):
        dd, got = self.dd, []
        for data, scoff in self.chunks[(self.seq // dd.nbatches) % NCHUNK]:
            with dd.get_input(self.seq) as slot:
                self.dequantize.launch(slot, scoff, data)
            with dd.get_output(self.seq) as out:
                got.append([out.out_max, out.out_argmax, out.out_score] if self.scored else [out.out_max, out.out_argmax])
            self.seq += 1
        return got


class GroupState:
    def __init__(self, case, seed):
        members = chains_of(case)
        self.group = pa.GpuDedisperserGroup([pa.DedispersionPlan(pa.DedispersionConfig.from_dict(config(m))) for m in members])
        self.group.allocate()
        self.dequantize, self.chunks = [], []
        for k, m in enumerate(members):
            fill_weights(self.group.members[k], m, seed + k)
            self.dequantize.append(pa.GpuDequantizationKernel(m['dtype'], m['beams'], sum(ints(m['nfreq'])), m['chunk']))
            self.chunks.append([packed_chunk(m, m['beams'], seed + k, c) for c in range(NCHUNK)])
        self.ichunk = 0
        for _ in range(NCHUNK - 1):
            self.one_chunk()

    def one_chunk(self):
        with self.group.get_input(self.ichunk) as slots:
            for kernel, chunks, slot in zip(self.dequantize, self.chunks, slots):
                data, scoff = chunks[self.ichunk % NCHUNK]
                kernel.launch(slot, scoff, data)
        with self.group.get_output(self.ichunk) as outs:
            got = [[o.out_max, o.out_argmax] for o in outs]
        self.ichunk += 1
        return got


class ScorerState:
    def __init__(self, case, seed):
        self.scorer = pa.LearnedScorer(params=network(seed))
        self.tiles, self.labels = tile_batch(case, seed)
        self.train = case['kind'] == 'train'

    def one_batch(self):
        s = self.scorer
        if not self.train:
            return s.forward(self.tiles)
        loss = s.train_step(self.tiles, self.labels, lr=2e-3)
        return {'loss': loss, 'grad': s.grad_buf, 'params': s.params, 'm': s.m, 'v': s.v}


def fill_weights(dd, case, seed):
    for it, t in enumerate(trees(case)):
        f, base = weight_factors(t, seed, it)
        w = f[:, :, None, None] * base[None, None, :, None]
        dd.fill_all_weights(it, np.broadcast_to(w, dd.wt_shape(it)))


def prepare(case, seed):
    if case['kind'] == 'chain':
        return ChainState(case, seed)
    if case['kind'] == 'group':
        return GroupState(case, seed)
    return ScorerState(case, seed)


def run(state):
    return state.one_batch() if isinstance(state, ScorerState) else state.one_chunk()


# ---------------------------------------------------------------------------------------------
# Compulsory work

def work(case):
    if case['kind'] in ('score', 'train'):
        n, size = case['tiles'], SIZE[case['dtype']]
        macs = COLS * TAPS * (CH * ROWS + 2 * CH * CH)
        if case['kind'] == 'score':
            return {'bytes': n * (ROWS * COLS * size + 4), 'flops': 2 * n * macs}
        back = COLS * TAPS * (CH * ROWS + 4 * CH * CH)      # weight gradients of 3 layers, data gradients of 2
        nparam = CH * ROWS * TAPS + 2 * CH * CH * TAPS + 5 * CH + 1
        return {'bytes': n * (ROWS * COLS * size + 8) + nparam * 4 * 8, 'flops': 2 * n * (macs + back)}
    nbytes = flops = 0
    for m in chains_of(case):
        B, F, T, size = m['beams'], sum(ints(m['nfreq'])), m['chunk'], SIZE[m['dtype']]
        nbytes += B * F * (T // 2 + T // 256 * 4)
        flops += B * 2 * T * (F + (1 << m['rank']))
        for p in range(len(ints(m['widths']))):      # the stage-1 outputs are kept for the rest of their delay
            nbytes += B * (T >> p) * (1 << (m['rank'] - (p > 0))) * size
            flops += B * (T >> p) * (2 << (m['rank'] - (p > 0))) * (m['rank'] // 2)
        for t in trees(m):
            nbytes += B * t['nt'] * (1 << t['tot']) * size          # and read once by each tree
            nbytes += B * t['ndm'] * t['nt_out'] * (size + 4) + B * t['ndm_wt'] * t['nt_wt'] * t['P'] * t['N'] * 4
            flops += B * t['nt'] * (2 << t['tot']) * (t['tot'] - t['tot'] // 2)
            cands = sum((t['dout'] // min(2 ** lev, min(t['dout'], 8))) * (3 if lev else 4)
                        for lev in range(max(1, (t['P'] - 1) // 3)))
            flops += B * t['ndm'] * t['M'] * t['nt_out'] * cands * 4
    return {'bytes': nbytes, 'flops': flops}


# ---------------------------------------------------------------------------------------------
# The same outputs in float64

def delayed(x, first):
    """x (bands, n, T): row d later by first + d samples, zeros before the start."""
    nb, n, T = x.shape
    pad = first + n - 1
    y = torch.zeros((nb, n, T + pad), dtype=x.dtype, device=x.device)
    y[:, :, pad:] = x
    return y.as_strided((nb, n, T), (n * (T + pad), T + pad - 1, 1), pad - first)


def combine(x, y, first):
    """Sums of neighbouring bands x (upper frequencies) and y over DM rows first, first + 1, ..."""
    c = math.sqrt(0.5)
    out = torch.empty((x.shape[0], x.shape[1], 2, x.shape[2]), dtype=x.dtype, device=x.device)
    torch.add(delayed(x, first), y, out=out[:, :, 0])
    torch.add(delayed(x, first + 1), y, out=out[:, :, 1])
    return out.mul_(c).view(x.shape[0], 2 * x.shape[1], x.shape[2])


def streams(t, rows):
    """Peak-finder streams of a tree: (subband n, rows (ndm, 2^level, time), final lag per DM row)."""
    a = rows[:1 << t['rr']].unsqueeze(1)
    first, n = 0, 0
    for r in range(t['rr']):
        lev = r + 1 + t['pf'] - t['rr']
        if lev == 1:                                        # the bands themselves, before the last pf passes
            for b in range(t['counts'][0]):
                yield n, a[b].unsqueeze(1), (1 << t['pf']) - (b + 1)
                n += 1
        if lev >= 1:
            for b in range(t['counts'][lev]):
                s = combine(a[b:b + 1], a[b + 1:b + 2], first)[0]
                fhi = b * (1 << (lev - 1)) + (1 << lev)
                yield n, s.view(t['ndm'], 1 << lev, -1), (1 << t['pf']) - fhi
                n += 1
        if r + 1 < t['rr']:
            a = combine(a[0::2], a[1::2], first)
            first *= 2
            if t['p'] > 0 and r == 0:                       # downsampled trees search the upper half of the DMs
                a, first = a[:, 1:].contiguous(), 1


def peaks(t, rows, weights, base):
    """(ndm, nt_out) largest weighted boxcar of the last chunk, and the full-band rows of it."""
    nt, W = t['nt'], t['width']
    margin = 4 * W
    best = rows_out = None
    dm = torch.arange(t['ndm'], device=rows.device) + (t['ndm'] if t['p'] else 0)
    win = torch.arange(nt + margin, device=rows.device) + rows.shape[1] - nt - margin
    wrow = torch.repeat_interleave(torch.repeat_interleave(weights, t['ndm'] // t['ndm_wt'], 0), t['nt_out'] // t['nt_wt'], 1)
    for _, s, lag in streams(t, rows):
        at = win[None, :] - lag * dm[:, None]
        x = torch.gather(s, 2, at.clamp(min=0)[:, None, :].expand(-1, s.shape[1], -1))
        x = torch.where((at >= 0)[:, None, :], x, torch.zeros((), dtype=x.dtype, device=x.device))
        rows_out = x[..., margin:]
        for lev in range(max(1, (t['P'] - 1) // 3)):
            w, dt = 1 << lev, min(1 << lev, min(t['dout'], 8))
            if lev:
                x = x + torch.nn.functional.pad(x, (w // 2, 0))[..., :x.shape[-1]]
            ends = torch.arange(dt, nt + 1, dt, device=rows.device) + margin - 1
            x3, x2, x1, x0 = (x[..., ends - k * w] for k in range(4))
            ys = [x3] if lev == 0 else [None]
            if t['P'] > 1:
                ys += [x2 + x3, 0.5 * x1 + x2 + 0.5 * x3, 0.5 * x0 + x1 + x2 + 0.5 * x3]
            for q, y in enumerate(ys):
                if y is not None:
                    y = y.reshape(t['ndm'], -1, t['nt_out'], t['dout'] // dt).amax(dim=(1, 3)) * wrow * base[3 * lev + q]
                    best = y if best is None else torch.maximum(best, y)
    return best, rows_out


def exact_beam(case, x, seed, outs, b, logits):
    """Fills beam b of each tree's out_max from its samples x (channels, time), float64."""
    f = channel_edges(case)
    n = np.arange((1 << case['rank']) + 1) / (1 << case['rank'])
    freq = (n * (f[0] ** -2.0 - f[-1] ** -2.0) + f[-1] ** -2.0) ** -0.5
    pos = np.clip(np.interp(freq, f, np.arange(len(f))), 0, len(f) - 1)
    low = np.minimum(pos.astype(np.int64), x.shape[0] - 1)
    total = torch.cat([torch.zeros_like(x[:1]), torch.cumsum(x, 0)])
    ilow = torch.from_numpy(low).to(x.device)
    total = total[ilow] + torch.from_numpy(pos - low).to(x.device)[:, None] * x[ilow]
    rows = (total[:-1] - total[1:]).contiguous()
    p = 0
    for it, t in enumerate(trees(case)):
        while p < t['p']:
            rows, p = (rows[:, 0::2] + rows[:, 1::2]) * math.sqrt(0.5), p + 1
        fac, base = weight_factors(t, seed, it)
        w = torch.from_numpy(fac.astype(np.float64)).to(x.device)
        outs[it][b], full = peaks(t, rows, w, [float(v) for v in base])
        if it == 0 and logits is not None:
            tiles = full.reshape(-1, ROWS, t['nt'] // COLS, COLS).transpose(1, 2).reshape(-1, ROWS, COLS)
            logits[b] = net(torch.from_numpy(network(seed)).to(x.device), tiles.contiguous()).view(logits[b].shape)


def samples(chunks, b):
    """float64 (channels, time) of beam b over the chunks."""
    xs = []
    for data, scoff in chunks:
        d = data[b].to(torch.int16)
        v = torch.stack([d & 15, d >> 4], dim=-1).view(d.shape[0], -1, 256)
        v = (v ^ 8) - 8
        s = scoff[b].double()
        xs.append(torch.where(v == -8, torch.zeros((), dtype=torch.float64, device=d.device),
                              s[..., 0:1] * v + s[..., 1:2]).view(d.shape[0], -1))
    return torch.cat(xs, 1)


def exact_chain(case, seed):
    chunks = [packed_chunk(case, case['beams'], seed, c) for c in range(NCHUNK)]
    ts = trees(case)
    outs = [torch.empty((case['beams'], t['ndm'], t['nt_out']), dtype=torch.float64, device=device()) for t in ts]
    logits = None
    if case['scorer']:
        logits = torch.empty((case['beams'], (1 << ts[0]['tot']) // ROWS, ts[0]['nt'] // COLS), dtype=torch.float64,
                             device=device())
    for b in range(case['beams']):
        exact_beam(case, samples(chunks, b), seed, outs, b, logits)
    got = []
    for i in range(0, case['beams'], case['batch']):
        one = [[o[i:i + case['batch']] for o in outs], [None] * len(outs)]
        got.append(one + [logits[i:i + case['batch']]] if case['scorer'] else one)
    return got


def net(params, tiles):
    """Logits of float64 tiles."""
    sizes = [CH * ROWS * TAPS, CH * CH * TAPS, CH * CH * TAPS, CH, CH, CH, CH, CH, 1]
    w1, w2, w3, b1, b2, b3, u, v, c0 = torch.split(params, sizes)
    a = tiles
    for w, b in ((w1, b1), (w2, b2), (w3, b3)):
        w = w.view(CH, -1, TAPS)
        x = torch.nn.functional.pad(a, (TAPS // 2, TAPS // 2))
        y = sum(torch.matmul(w[:, :, k].contiguous(), x[:, :, k:k + COLS].contiguous()) for k in range(TAPS))
        a = torch.relu(y + b[:, None])
    return c0 + a.amax(2) @ u + a.mean(2) @ v


def exact_scorer(case, seed):
    params = torch.from_numpy(network(seed)).to(device())
    tiles, y = tile_batch(case, seed)
    n, y = case['tiles'], y.double()
    if case['kind'] == 'score':
        return torch.cat([net(params, tiles[i:i + 512].double()) for i in range(0, n, 512)])
    params.requires_grad_(True)
    loss, grad = 0.0, torch.zeros_like(params)
    for i in range(0, n, 512):
        z = net(params, tiles[i:i + 512].double())
        part = torch.nn.functional.binary_cross_entropy_with_logits(z, y[i:i + 512], reduction='sum') / n
        grad += torch.autograd.grad(part, params)[0]
        loss = loss + part.detach()
    m, v = 0.1 * grad, 0.001 * grad * grad
    new = params.detach() - 2e-3 * (m / 0.1) / (torch.sqrt(v / 0.001) + 1e-8)
    return {'loss': loss, 'grad': grad, 'params': new, 'm': m, 'v': v}


def exact(case, seed):
    if case['kind'] == 'chain':
        return exact_chain(case, seed)
    if case['kind'] == 'group':
        got = [exact_chain(m, seed + k)[0] for k, m in enumerate(chains_of(case))]
        return got
    return exact_scorer(case, seed)
