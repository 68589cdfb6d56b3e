"""What a part may see of the running step, and the scratch memory it may use."""
from __future__ import annotations

import ctypes

import torch

from ..kernels.ops import PinnedCopy


class Workspace:
    """Named scratch buffers that live as long as the runner.  `reserve` carves every buffer that the
    parts have named for the largest step out of ONE allocation; a name that was not planned (a part
    without a plan), or a size beyond its plan, is allocated when it is first asked for and grows only
    when a larger size is asked, so steady steps allocate nothing either way.  The buffers of COUNTERS hold zeros when they are
    made; whoever counts in one leaves zeros behind."""

    COUNTERS = ("arrivals",)

    def __init__(self, device):
        self.device = torch.device(device)
        self._buffers = {}
        self._arena = None
        self.planned_bytes = 0
        self._unplanned = {}          # (name, dtype) -> bytes allocated outside the plan
        self._views = {}              # (name, dtype, shape) -> the view handed out for it

    @staticmethod
    def plan_bytes(plan):
        """plan: {(name, dtype): elements}.  Bytes of the one allocation that holds them (256-byte places)."""
        return sum(-(-count * torch.empty((), dtype=dtype).element_size() // 256) * 256
                   for (_, dtype), count in plan.items())

    def reserve(self, plan):
        total = self.plan_bytes(plan)
        self._arena = torch.empty(max(total, 1), dtype=torch.uint8, device=self.device)
        self.planned_bytes = total
        at = 0
        for (name, dtype), count in plan.items():
            size = count * torch.empty((), dtype=dtype).element_size()
            self._buffers[(name, dtype)] = self._arena[at:at + size].view(dtype)
            if name in self.COUNTERS:
                self._buffers[(name, dtype)].zero_()
            at += -(-size // 256) * 256

    def unplanned_bytes(self):
        return sum(self._unplanned.values())

    def get(self, name, shape, dtype):
        # (a step asks for the same few shapes again and again: the views are kept, a steady step makes none)
        shape = tuple(shape)
        view = self._views.get((name, dtype, shape))
        if view is not None:
            return view
        count = 1
        for extent in shape:
            count *= int(extent)
        key = (name, dtype)
        buf = self._buffers.get(key)
        if buf is None or buf.numel() < count:
            buf = (torch.zeros if name in self.COUNTERS else torch.empty)(max(count, 1), dtype=dtype, device=self.device)
            self._buffers[key] = buf
            self._unplanned[key] = buf.numel() * buf.element_size()
            for stale in [k for k in self._views if k[0] == name and k[1] == dtype]:
                del self._views[stale]                     # (views of the buffer that this one replaces)
        view = buf[:count].view(shape)
        if len(self._views) >= 4096:
            self._views.clear()
        self._views[(name, dtype, shape)] = view
        return view

    def room(self, name, dtype):
        """Elements that the name's buffer holds now."""
        buf = self._buffers.get((name, dtype))
        return 0 if buf is None else buf.numel()

    def bytes(self):
        return self.planned_bytes + self.unplanned_bytes()

    def buffers(self):
        """The buffers as they are now.  A captured graph holds on to this list: it keeps using the
        memory it was captured with, also after a larger step has made a name's buffer grow."""
        return list(self._buffers.values())


class Uploader:
    """Small host-to-device copies through one pinned buffer.  The copy is asynchronous; an event
    guards the buffer so that the next use waits until the previous copy has left it."""

    def __init__(self, capacity, device):
        self.device = torch.device(device)
        self._copy = PinnedCopy()
        self._reserve(capacity)

    def _reserve(self, capacity):
        self._host = torch.empty(capacity, dtype=torch.int32).pin_memory()
        self._view = self._host.numpy()
        self.address = ctypes.c_void_p(self._host.data_ptr())

    def stage(self, n):
        """The buffer's first n values as an int32 numpy vector, free to be written."""
        self._copy.wait()
        if n > self._view.size:
            self._reserve(max(n, 2 * self._view.size))
        return self._view[:n]

    def upload(self, n, dst):
        """The first n values to the device int32 vector dst, which holds at least that many."""
        self._copy.copy(dst, self.address, 4 * n)

    def send(self, values, dst):
        """values: a list of ints or an int32 numpy vector; dst: device int32 vector of at least that many elements."""
        n = len(values)
        self.stage(n)[:] = values
        self.upload(n, dst)


# Single tokens that fill the GPU without a split, one workgroup a token and kv head: the longest context of the batch would
# keep its workgroup walking when the others are done, so no workgroup walks more than this many keys.  Measured with 64
# requests of 129 to 3001 tokens: a step of the 0.6B sizes 3.69 ms instead of 4.25 (ranges of 1024: 3.79), of four layers of the
# 8B sizes 1.30 instead of 1.41; with 64 requests of 3900 tokens each, where a split only adds partial results, 6.90 instead of
# 6.87 and 1.71 instead of 1.69.
LONG_RANGE = 2048


class StepContext:
    """One step's view for the parts: the tokens with their positions and slots (device int32
    vectors of equal length), the segments they form (host), the cache, the kernels and the
    scratch memory."""

    def __init__(self, kernels, cache, workspace, dtype, max_positions, split_keys, split_max_tokens):
        self.kernels, self.cache, self.workspace, self.dtype = kernels, cache, workspace, dtype
        self.max_positions = max_positions
        self.split_keys, self.split_max_tokens = split_keys, split_max_tokens
        self.target_workgroups = 512      # about two workgroups per compute unit
        self.compute_units = (torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
                              if torch.cuda.is_available() else 1)
        self.n_tokens = 0
        self.token_ids = self.positions = self.slots = None
        self.segments = []            # (slot, first row, number of tokens, first position)
        self.state_rows = None        # device int32, a value a token: its request's live row of the paired entries (where there are any)
        self.segment_slots = None     # device int32, one slot per segment (set when the model keeps state per request)
        self.single_tokens = False    # every segment brings exactly one token (a decoding step)
        self.max_context = 0          # largest position + 1 among the step's tokens
        self._groups = {}
        self._left_out = {}           # buffer of token groups without some entries -> the sets of entries it was asked without
        self._group_upload = None
        self.fixed_groups = None      # a captured step's groups: {key: token_groups' result}, in tensors of their own
        self.status = None            # device int32 [2] when the hidden state is to be checked after every layer
        self.partial_budget = None    # floats that split attention's partial results may take (the memory plan's)
        self.routed = False           # the model chooses among experts (`DecoderModel.routes`)

    def begin_step(self):
        self._groups, self._left_out = {}, {}
        self.fixed_groups = None

    def token_groups(self, tokens_per_group, big_factor=0, without=(), rest="rest"):
        """The step's rows cut into groups of consecutive tokens of one request, as device int32 vectors
        (first row of each group, tokens in each group) with their number.  Returns (small, big, (rows in
        small groups, one beyond the last batch row of a small group)): small groups hold at most
        `tokens_per_group` tokens; with big_factor > 0, a request that brings more than `tokens_per_group`
        tokens is cut into big groups of at most big_factor * tokens_per_group instead (prompt portions), else
        `big` is empty.  `without`: entries of the step (their numbers, ascending) whose rows are left out; `rest` then
        ends the name of the buffer, for callers that leave out different entries of one step (a buffer asked again without
        other entries gets another one beside it: what was handed out before stays as it is)."""
        key = (tokens_per_group, big_factor, without)
        hit = self._groups.get(key)
        if hit is not None:
            return hit
        if self.fixed_groups is not None and key in self.fixed_groups:
            return self.fixed_groups[key]
        first, count, big_first, big_count = [], [], [], []
        small_rows = small_end = 0
        for i, (_, row, n, _) in enumerate(self.segments):
            if i in without:
                continue
            if big_factor > 0 and n > tokens_per_group:
                size = big_factor * tokens_per_group
                for at in range(0, n, size):
                    big_first.append(row + at)
                    big_count.append(min(size, n - at))
            else:
                small_rows += n
                small_end = max(small_end, row + n)
                for at in range(0, n, tokens_per_group):
                    first.append(row + at)
                    count.append(min(tokens_per_group, n - at))
        g, gb = len(first), len(big_first)
        if self.fixed_groups is not None:
            # a step that is to be captured: its groups depend on the lengths of its entries only, so they
            # get a tensor of their own once (this is the eager run before the capture) and stay there
            dev = torch.tensor(first + count + big_first + big_count + [0], dtype=torch.int32, device=self.workspace.device)
        else:
            name = f"token_groups_{tokens_per_group}_{big_factor}"
            if without:
                name = f"{name}_{rest}"
                sets = self._left_out.setdefault(name, [])
                if without not in sets:
                    sets.append(without)
                if sets.index(without) > 0:
                    name = f"{name}_{sets.index(without)}"
            dev = self.workspace.get(name, (2 * (g + gb),), torch.int32)
            if self._group_upload is None:
                self._group_upload = Uploader(4096, dev.device)
            self._group_upload.send(first + count + big_first + big_count, dev)
        hit = ((dev[:g], dev[g:2 * g], g), (dev[2 * g:2 * g + gb], dev[2 * g + gb:2 * g + 2 * gb], gb),
               (small_rows, small_end))
        if self.fixed_groups is not None:
            self.fixed_groups[key] = hit
        self._groups[key] = hit
        return hit

    def attention_split(self, rows, batch_rows, kv_heads, q_heads, head_dim, longest=None, narrow=True):
        """(split_keys, max_splits, partial buffer).  A batch of many tokens fills the GPU with one
        workgroup per (token group, kv head); a small batch over long contexts does not, so there the
        keys of a token are split over several workgroups, in ranges [s * split_keys, (s + 1) *
        split_keys) of absolute key positions, and merged in ascending order.  split_keys is the
        largest of base, 2 base, 4 base, ... that still gives `target_workgroups`, or where base is too wide for that narrower
        (`narrowed`; not in a model that routes, whose choices turn on the last bit, nor where `narrow` says no); what a token's
        result is does not depend on the choice beyond rounding.  `rows` tokens take part; the partial
        results are indexed by batch row, of which there are `batch_rows`.  `longest`: the most keys a
        workgroup of the kernel can walk without a split; a longer context is split whatever the batch."""
        forced = longest is not None and self.max_context > longest
        if rows > self.split_max_tokens and not forced:
            return 0, 1, None
        return self._split(max(1, rows * kv_heads), self.target_workgroups, batch_rows, q_heads, head_dim, longest, LONG_RANGE,
                           narrow=narrow and not self.routed)

    def even_split(self, rows, kv_heads, q_heads, head_dim):
        """(workgroups, wide, max_splits, partial buffer) for single tokens whose key ranges are merged in the launch that makes them
        (`attention_decode_fused`): every token's keys in ranges of its own, evenly wide (`even_ranges`); None where `attention_split`
        has to say: no splits wanted, a model that routes, partial results that would not fit, so many tokens that one has not two units.

        One workgroup a compute unit takes the keys as fast as two, each more is another partial result that the merge waits for, and a
        few more than fill the units cost a second round.  Measured with 1 to 64 tokens of 16 query and 8 kv heads of 128 channels behind
        400 to 8000 keys, pages cold, us a layer, ranges as `attention_split` cuts them and even ones: 1 token behind 1100 keys 12.6, 12.2;
        behind 3800 15.1, 15.3; 2 behind 1100 15.9, 12.9; 6 behind 2000 21.4, 20.1; 8 behind 4600 to 4900 43.2, 40.1; 12 behind 2000
        30.9, 28.0; 16 behind up to 3800 38.8, 37.4.  Not beyond half the units: 24 behind 2000 50.7, 45.0, but 24 behind 300 to 3800 48.5,
        59.2, where a long context's one range keeps the step waiting, and 64 behind 129 to 3000, whose second ranges are dealt out when
        the first are done, 76.3, 84.6.  Longer contexts, where a token has two to four shares of ranges: 1 token behind 16300 24.1, 20.6, behind
        40000 45.8, 36.6; 4 behind 32768 113.3, 113.8, 40000 138.5, 126.4; 8 behind 16300 100.8, 100.6, 32768 205.3, 198.5, 40000 253.3, 243.5; 16 behind
        24576 308.6, 293.4, 32768 401.1, 395.1.  (4 behind 8100 31.9, 35.6, where ranges lie 1024 keys apart, it seems on the same channels of memory; 4
        behind 8300, 1088 keys each, 34.2, 31.6.)"""
        units, workgroups = rows * kv_heads, min(self.compute_units, self.target_workgroups)
        if rows > self.split_max_tokens or self.split_keys <= 0 or self.routed or 2 * units > workgroups:
            return None
        wide = -(-LONG_RANGE * workgroups // units // 64) * 64
        max_splits = self.even_ranges(self.max_context, workgroups, units, wide)
        numel = self.kernels.attention_partial_numel(rows, q_heads, head_dim, max_splits)
        if max_splits > 1024 or (self.partial_budget is not None and numel > self.partial_budget):
            return None
        return workgroups, wide, max_splits, self.workspace.get("attn_partial", (numel,), torch.float32)

    @staticmethod
    def even_ranges(walk, workgroups, units, wide):
        """The kernel's rule (`even_ranges` in attention.hip) for one token behind `walk` keys: it never gives a shorter context more
        ranges than a longer one."""
        return max(1, min(workgroups * -(-walk // wide) // units, max(16, walk // 256), -(-walk // 64)))

    def group_split(self, groups, batch_rows, kv_heads, q_heads, head_dim, longest=None):
        """As `attention_split` for `groups` groups of many tokens each (prompt portions), which give
        one workgroup per (group, kv head).  `longest`: the most keys a workgroup can take without a
        split; a longer context is split whatever the number of groups."""
        return self._split(max(1, groups * kv_heads), self.compute_units, batch_rows, q_heads, head_dim, longest)

    def fixed_split(self, rows, q_heads, head_dim):
        """(split_keys, max_splits, rows a launch, partial buffer) for the attention kernel whose results must
        not depend on the batch by a single bit (the float engine's): a token's keys are always cut into ranges
        of `split_keys` of the runner's setting, whatever else the step holds, so the sums that make up its
        result and their order follow from its own position alone.  (A context of more than 1024 ranges
        doubles their width: the merge kernel's limit.)  The partial results of all rows may exceed what was
        planned for them; then the rows are served by several launches."""
        base = self.split_keys
        if base <= 0 or self.max_context <= base:
            return 0, 1, rows, None
        keys = base
        while -(-self.max_context // keys) > 1024:
            keys *= 2
        max_splits = -(-self.max_context // keys)
        per_row = self.kernels.attention_partial_numel(1, q_heads, head_dim, max_splits)
        chunk = rows if self.partial_budget is None else max(1, min(rows, self.partial_budget // per_row))
        return keys, max_splits, chunk, self.workspace.get("attn_partial", (chunk * per_row,), torch.float32)

    @staticmethod
    def narrowed(base, walk, units, enough, ranges):
        """The width of a key range where ranges of `base` keys leave the chip idle, `units` workgroups a range, for contexts of up to
        `walk` keys: halved, to 64 keys at least, while that gives no more than `enough` workgroups and `ranges` ranges.  A
        workgroup's time is a chain of tiles, the merge's a chain of ranges, sixteen of which it asks for at once.

        Plain attention, weights cold: one request of the 0.6B sizes behind 200, 700, 1100 and 1500 tokens 1173, 1175, 1175 and 1182 us a
        step with ranges of 256, now 1088, 1098, 1128 and 1140; three of four 8B layers behind 700 to 1200 669 -> 647.  Behind 3900 tokens
        32 ranges would cost 6 %; four requests of 1000 to 1900 tokens on 512 workgroups, two a compute unit, 5 % (400: as before).
        Differential attention, where half a workgroup works, gains up to 512 and 32 ranges: 8 requests of 1000 to 1700 tokens 714 -> 683."""
        keys = base
        while keys % 128 == 0 and -(-walk // (keys // 2)) <= ranges and units * -(-walk // (keys // 2)) <= enough:
            keys //= 2
        return keys

    @staticmethod
    def forced_splits(max_length, base, longest):
        """Key splits that a context of `max_length` needs at least when one workgroup walks at most `longest`
        keys: ranges of the largest of base, 2 base, 4 base, ... that `longest` holds (1: no split needed)."""
        if longest is None or max_length <= longest or base <= 0:
            return 1
        keys = base
        while keys * 2 <= longest:
            keys *= 2
        return -(-max_length // keys)

    def _split(self, units, enough, batch_rows, q_heads, head_dim, longest=None, widest=None, narrow=False):
        """`units` workgroups without a split; no split when they are `enough`, but for contexts beyond `widest` keys.  The partial results never take
        more than `partial_budget` floats (when one is set: the runner's memory plan): key ranges are doubled
        until they fit, which a forced split allows up to `longest`."""
        base = self.split_keys
        forced = longest is not None and self.max_context > longest
        if base <= 0 or (self.max_context <= base and not forced):
            return 0, 1, None
        keys = self.narrowed(base, self.max_context, units, 3 * self.compute_units // 2, 20) if narrow else base
        while keys * 2 < self.max_context and units * (-(-self.max_context // (keys * 2))) >= self.target_workgroups:
            keys *= 2
        if forced:
            while keys > base and keys > longest:
                keys //= 2
        elif units >= enough:
            if widest is None or self.max_context <= widest:
                return 0, 1, None
            while keys < widest:
                keys *= 2
            while keys > base and keys > widest:
                keys //= 2
        budget = self.partial_budget
        numel = lambda k: self.kernels.attention_partial_numel(batch_rows, q_heads, head_dim, -(-self.max_context // k))
        while budget is not None and numel(keys) > budget and (not forced or keys * 2 <= longest):
            if keys >= self.max_context:                 # one range holds every key: no split, nothing to keep
                return 0, 1, None
            keys *= 2
        max_splits = -(-self.max_context // keys)
        if max_splits <= 1:
            return 0, 1, None
        while max_splits > 1024:                     # the merge kernels' limit
            keys *= 2
            max_splits = -(-self.max_context // keys)
        numel = self.kernels.attention_partial_numel(batch_rows, q_heads, head_dim, max_splits)
        return keys, max_splits, self.workspace.get("attn_partial", (numel,), torch.float32)
