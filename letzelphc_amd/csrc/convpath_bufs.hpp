// convpath_bufs.hpp -- device buffers of the sphere form (convpath.hpp).
// Included by lelph_hip.hip before the context, which owns a set.
#pragma once

// working buffers of one stream of groups
struct ConvBufs
{
    DBuf desc, map, coef, line, box, c, part;
    void release()
    {
        for (DBuf* b : {&desc, &map, &coef, &line, &box, &c, &part}) b->release();
    }
};
