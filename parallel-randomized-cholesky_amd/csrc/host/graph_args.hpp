// graph_args.hpp -- what a captured graph was recorded with.
//
// A captured launch keeps its arguments by value: pointers, counts and grids.
// A cached graph may run again only with the very same ones.  Comparing them
// whole leaves no buffer out that can move, or size that can change, on its own.
#pragma once

#include <cstring>
#include <type_traits>

template <typename A>
class GraphArgs {
    static_assert(std::is_trivially_copyable_v<A> && std::has_unique_object_representations_v<A>,
                  "compared by bytes: no padding");

public:
    bool same(const A &b) const { return set_ && std::memcmp(&a_, &b, sizeof(A)) == 0; }
    void set(const A &b)
    {
        std::memcpy(&a_, &b, sizeof(A));
        set_ = true;
    }

private:
    A a_{};
    bool set_ = false;
};
