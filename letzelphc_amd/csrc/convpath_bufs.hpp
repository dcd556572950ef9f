// convpath_bufs.hpp -- device buffers of the sphere form (convpath.hpp) and of
// the non-local part (nlpath.hpp).
// Included by lelph_hip.hip before the context, which owns a set.
#pragma once

// Grows b to need bytes; work on st that may still use it ends first.  fixed:
// uploaded descriptors that are run again (a captured pass) hold b's address,
// so it must be large enough already.
static int buf_grow(DBuf& b, size_t need, bool fixed, hipStream_t st)
{
    if (need <= b.n) return LELPH_OK;
    if (fixed) return LELPH_ERR_STATE;
    if (b.p) HIP_TRY(hipStreamSynchronize(st));
    return b.ensure(need);
}

// working buffers of one stream of groups
struct ConvBufs
{
    DBuf desc, map, coef, line, box, c, part;
    bool fixed = false; // sized for every group that uses them (conv_reserve)
    void release()
    {
        for (DBuf* b : {&desc, &map, &coef, &line, &box, &c, &part}) b->release();
    }
};

// non-local part: scratch of the sides formed together, their projections,
// the K/K' sums of a group of pairs, bf16 pieces (nl_form 1)
struct NlBufs
{
    DBuf desc, side, bb, ebuf, splitA, splitB;
    bool fixed = false; // sized for every window that uses them (nl_reserve)
    const int* kk = nullptr; // pairs' key numbers of the current window
    void release()
    {
        for (DBuf* b : {&desc, &side, &bb, &ebuf, &splitA, &splitB}) b->release();
    }
};

// the sides and pairs of one window: keys in order of first use, two key
// numbers (k+q, k) per pair
struct NlWindow
{
    std::vector<std::array<int, 2>> keys; // (iBZ k, symmetry)
    std::vector<int> kk;
    void add(const lelph_pair& p)
    {
        kk.push_back(key(p.ikq, p.kqsym));
        kk.push_back(key(p.ik, p.ksym));
    }

  private:
    std::map<std::array<int, 2>, int> at;
    int key(int ik, int sym)
    {
        const std::array<int, 2> k = {ik, sym};
        const auto r = at.insert({k, (int)keys.size()});
        if (r.second) keys.push_back(k);
        return r.first->second;
    }
};
