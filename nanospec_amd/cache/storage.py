"""The memory behind the cache manager: pages of keys and values per group of layers, and state slots.

A run-order entry of the model with a ``PagedNeed`` gets one layer of its group's page tensors:
    K [entries, pages, kv_heads, page, head_dim]       (the reference keeps [pages, page, kv_heads, head_dim],
                                                        kv/cache.py:16-19; here a head's part of a page is contiguous)
    V [entries, pages, kv_heads, value_dim, page]      (transposed per page for the attention kernels; value_dim is
                                                        head_dim unless the mixer says otherwise)
Both start as zeros: slots that are masked out are still read (reference: kv/cache.py:18).  A page id
means the same page in every entry of its group.  An entry with a ``StateNeed`` gets a tensor
[slots, *shape]; an entry that reads another entry's cache gets that entry's view.
"""

from __future__ import annotations

from dataclasses import dataclass

import torch

from ..kernels.ops import SlotTensors
from ..parts.needs import PagedNeed, StateNeed, each_need
from .manager import GroupSpec


STEPS_SHARE = 0.1  # of the device's memory that is to be left for the steps beside weights, pages and states


@dataclass
class PagedView:
    group: int
    k: torch.Tensor
    v: torch.Tensor


@dataclass
class StateView:
    state: torch.Tensor  # [slots, *shape]


def plan_groups(cache_needs: list) -> tuple[list[GroupSpec], list[PagedNeed], list[int | None]]:
    """Run-order entries with equal paged needs share a group.  -> (group specs for the manager, the need
    of each group, group index of each entry or None)."""
    needs: list[PagedNeed] = []
    of_entry: list[int | None] = []
    for need in cache_needs:
        if isinstance(need, PagedNeed):
            if need not in needs:
                needs.append(need)
            of_entry.append(needs.index(need))
        else:
            # (an entry whose mixer is made of several: its paged needs join their groups; ``of_entry`` names the first)
            first = None
            for single in each_need(need) if isinstance(need, (tuple, list)) else ():
                if isinstance(single, PagedNeed):
                    if single not in needs:
                        needs.append(single)
                    first = needs.index(single) if first is None else first
            of_entry.append(first)
    specs = [GroupSpec(n.group_name, n.window) for n in needs]
    return specs, needs, of_entry


class CacheStorage:
    def __init__(self, model, num_pages: list[int], page_size: int, num_slots: int, dtype, device) -> None:
        # what a model keeps only to be faster makes room: where the pages do not fit beside it, or leave little for the steps
        give_back = getattr(model, "give_back_second_copies", lambda: False)
        short = False
        try:
            self._allocate(model, num_pages, page_size, num_slots, dtype, device)
        except torch.OutOfMemoryError:
            short = True
        if short:  # (behind the handler, whose traceback holds what had been allocated)
            self.__dict__.clear()
            give_back()
            self._allocate(model, num_pages, page_size, num_slots, dtype, device)
        elif dtype == torch.float32 and torch.device(device).type == "cuda":  # (no other models have such copies)
            free, total = torch.cuda.mem_get_info(device)
            if free + torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device) < STEPS_SHARE * total:
                give_back()

    def _allocate(self, model, num_pages: list[int], page_size: int, num_slots: int, dtype, device) -> None:
        self.group_specs, needs, of_entry = plan_groups(model.cache_needs)
        self.page_size = page_size
        flat = [(single, i) for i, (need, call) in enumerate(zip(model.cache_needs, model.spec.run_order)) if call.cache_from is None
                for single in each_need(need)]
        counts = [sum(1 for single, _ in flat if isinstance(single, PagedNeed) and needs.index(single) == i) for i in range(len(needs))]
        self.k = [torch.zeros((counts[i], num_pages[i], n.kv_heads, page_size, n.head_dim), dtype=dtype, device=device)
                  for i, n in enumerate(needs)]
        self.v = [torch.zeros((counts[i], num_pages[i], n.kv_heads, n.v_dim, page_size), dtype=dtype, device=device)
                  for i, n in enumerate(needs)]
        self.states: list[torch.Tensor] = []
        self.views: list = []
        taken = [0] * len(needs)
        def view_of(need):
            if isinstance(need, (tuple, list)):
                return tuple(view_of(single) for single in need)
            if isinstance(need, PagedNeed):
                g = needs.index(need)
                view = PagedView(g, self.k[g][taken[g]], self.v[g][taken[g]])
                taken[g] += 1
                return view
            if isinstance(need, StateNeed):
                t = torch.zeros((num_slots, *need.shape), dtype=need.dtype, device=device)
                self.states.append(t)
                return StateView(t)
            return None

        for i, (need, call) in enumerate(zip(model.cache_needs, model.spec.run_order)):
            self.views.append(self.views[call.cache_from] if call.cache_from is not None else view_of(need))
        # state that belongs to the model and to no layer (``model.state_needs``: name -> StateNeed)
        self.model_state: dict[str, torch.Tensor] = {}
        for name, need in getattr(model, "state_needs", {}).items():
            t = torch.zeros((num_slots, *need.shape), dtype=need.dtype, device=device)
            self.states.append(t)
            self.model_state[name] = t
        # (a single state is as fast through its own fill, and the CPU has no launches to save)
        self._slots = SlotTensors(self.states) if len(self.states) > 1 and torch.device(device).type == "cuda" else None

    def reset_slot(self, slot: int) -> None:
        """A newly admitted request starts from zero state."""
        if self._slots is not None:
            self._slots.clear(slot)
            return
        for t in self.states:
            t[slot].zero_()

    def bytes_per_token(self) -> int:
        return sum((k[:, 0, :, 0].numel() + v[:, 0, :, :, 0].numel()) * k.element_size() for k, v in zip(self.k, self.v))
