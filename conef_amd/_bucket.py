"""Small helpers shared by the hooks: GradBucket accessors that accept both the current
torch spelling (buffer/gradients/index/is_last) and the one the reference was written against
(get_tensor/get_per_parameter_tensors/get_index/is_the_last_bucket_to_allreduce, e.g.
communication/powerSGD_hook.py:343,386,355,244), and a completed Future."""
import torch
import torch.distributed as dist

from . import _host


def buffer(bucket):
    return (getattr(bucket, "buffer", None) or bucket.get_tensor)()


def gradients(bucket):
    return (getattr(bucket, "gradients", None) or bucket.get_per_parameter_tensors)()


def index(bucket):
    return (getattr(bucket, "index", None) or bucket.get_index)()


def is_last(bucket):
    return (getattr(bucket, "is_last", None) or bucket.is_the_last_bucket_to_allreduce)()


def layout(grads):
    """What a step asks (``layout(grads)(grads_now)``) to see that a bucket still has the tensors its cached
    tables were made for: the shape of every one, in order.  The buffer's place and length go into the cache
    keys beside it."""
    return _host.same_shapes(grads)


def draw_starts(rng, numels, items, starts):
    """Block starts for the tensors of a bucket, one draw each, into the item table (``starts`` is the view
    of its start fields).  RandomState.choice(n) of an int n draws randint(0, n); randint over an array of
    bounds draws the same numbers from the same stream, one after the other, for 6 us a call against 1.5 us
    a number: the array from five tensors on."""
    if len(numels) < 5:
        for it, numel in zip(items, numels):
            it.start = int(rng.randint(0, numel))
    else:
        starts[:] = rng.randint(0, numels)


def group_and_size(process_group):
    """(group, world_size).  Without an initialised process group the world is one rank."""
    if process_group is not None:
        return process_group, process_group.size()
    if dist.is_available() and dist.is_initialized():
        return dist.group.WORLD, dist.group.WORLD.size()
    return None, 1


def completed_future(tensor):
    """A Future already holding ``tensor``; aware of the tensor's device so that DDP orders its
    own stream after the kernels enqueued by the hook."""
    fut = torch.futures.Future(devices=[tensor.device]) if tensor.is_cuda else torch.futures.Future()
    fut.set_result(tensor)
    return fut


def allreduce_fut(group, tensor, world_size):
    """Averaging all-reduce as a Future (what default._allreduce_fut does in the reference).
    At world size 1 the sum is the tensor itself and the division is by one."""
    if world_size == 1:
        return completed_future(tensor)
    tensor.div_(world_size)
    return dist.all_reduce(tensor, group=group, async_op=True).get_future().then(lambda f: f.value()[0])
