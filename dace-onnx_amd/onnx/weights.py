"""The weights of a model, and which of them a copy in another layout can stand for."""


class Weights(dict):
    """Weight name -> tensor.

    Launches read a weight where it lies, so that whatever was written into it takes effect: by torch, which counts some of that, through
    ``Tensor.data`` or by another library, which it does not. A packed copy is as good only while nobody else can write the weight, that
    is for tensors that the model made itself: the copies that fusion derives, which are its own, and the initializers it uploaded, until
    they are handed out. Reading an entry hands it out.
    """

    def __init__(self):
        super().__init__()
        self._made, self._derived, self._handed_out = {}, set(), set()

    def make(self, name, tensor, derived=False):
        """Add a tensor that nobody else holds."""
        self[name] = self._made[name] = tensor
        if derived:
            self._derived.add(name)

    def peek(self, name):
        """The tensor, for readers inside the package that do not keep it; None if there is none."""
        return dict.get(self, name)

    def peek_items(self):
        return dict.items(self)

    def derived(self, name):
        return name in self._derived

    def private(self, name):
        """Whether the entry is a tensor that only the model writes."""
        made = self._made.get(name)
        return made is not None and dict.get(self, name) is made and (name in self._derived or name not in self._handed_out)

    # -- every way to read an entry; the iterator is named so that dict(w), {**w} and f(**w) read entry by entry
    def __iter__(self):
        return super().__iter__()

    def __getitem__(self, name):
        self._handed_out.add(name)
        return super().__getitem__(name)

    def get(self, name, default=None):
        self._handed_out.add(name)
        return super().get(name, default)

    def setdefault(self, name, default=None):
        self._handed_out.add(name)
        return super().setdefault(name, default)

    def pop(self, name, *default):
        self._handed_out.add(name)
        return super().pop(name, *default)

    def popitem(self):
        self._handed_out.update(self)
        return super().popitem()

    def items(self):
        self._handed_out.update(self)
        return super().items()

    def values(self):
        self._handed_out.update(self)
        return super().values()

    def copy(self):
        return dict(self)

    def __or__(self, other):
        return dict(self) | other
