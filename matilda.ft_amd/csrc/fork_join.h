// Work spread over side streams between a fork from one stream and a join back
// to it, whatever fails in between.
#pragma once

namespace mft {

// work(g, k) queues item g of n on stream k = g % nstreams; stream 0 is the one
// that is forked from.  fork(k) makes stream k wait for stream 0 and join(k)
// makes stream 0 wait for stream k; each returns 0 or an error.  Every stream
// whose fork succeeded is joined, also after an error: later work on stream 0
// (new fields, a replica's reset, the frees of a teardown behind its
// synchronisation) then comes after all that was queued, and a capture of
// stream 0 ends with no stream left in it.  Returns the first error.
template <class Fork, class Work, class Join>
int fork_join(int nstreams, int n, Fork fork, Work work, Join join)
{
    int rc = 0, forked = 1;
    while (!rc && forked < nstreams)
        if (!(rc = fork(forked))) ++forked;
    for (int g = 0; !rc && g < n; ++g) rc = work(g, g % nstreams);
    for (int k = 1; k < forked; ++k) {
        const int r = join(k);
        if (!rc) rc = r;
    }
    return rc;
}

} // namespace mft
