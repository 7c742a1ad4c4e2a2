// What a test needs to see of a finalized program: its operations with the addresses that they read and write, and the
// order that the streams and events give them.
#include <stdio.h>
#include <string.h>

#include <string>

#include "hip/hip_common.hpp"

using namespace saga;

static HipProgram *program(void *box) { return dynamic_cast<HipProgram *>(((std::shared_ptr<Program> *)box)->get()); }

static std::string touched(const HipOpArgs &args)
{
    std::string r;
    for(const auto &a : args) {
        HipStorage *s = a.second->m_storage.get();
        // (a batched tensor has two addresses that belong to it alone; memory that nobody has asked for yet has none)
        const bool own = s->doubleBuffered() || !s->allocated();
        r += fmt("%s[%d,%llu,%zu,\"%s\"]", r.empty() ? "" : ",", s->m_id, (unsigned long long)(own ? 0 : (uintptr_t)s->m_data), s->bytes(),
                 a.first);
    }
    return r;
}

extern "C" {

// One line of JSON per operation.  fork: the operation of the main stream that one on the side stream waits for, -1 for the
// start of the step; needs: the operation of the side stream that one of the main stream waits for.  recorded: whether its launches
// go into a graph; safe: whether they may.
int probe_plan(void *box, char *buf, size_t capacity)
{
    HipProgram *p = program(box);
    const auto &side = p->m_side;
    std::string out;
    for(size_t i = 0; i < p->m_ops.size(); i++) {
        int fork = -1, needs = -1;
        if(i < side.size())
            for(size_t j = 0; j < side.size(); j++) {
                if(side[i].on && side[i].fork == side[j].reached && side[j].reached)
                    fork = (int)j;
                if(side[i].needs && side[i].needs == side[j].done)
                    needs = (int)j;
            }
        bool recorded = false;
        for(const auto &sg : p->m_segments)
            recorded |= sg.graph && sg.begin <= i && i < sg.end;
        out += fmt("{\"kind\":\"%s\",\"side\":%d,\"fork\":%d,\"needs\":%d,\"recorded\":%d,\"safe\":%d,\"reads\":[%s],\"writes\":[%s]}\n",
                   p->m_ops[i]->name().c_str(), i < side.size() && side[i].on ? 1 : 0, fork, needs, recorded ? 1 : 0,
                   p->m_ops[i]->graphSafe() ? 1 : 0, touched(p->m_ops[i]->getInputs()).c_str(),
                   touched(p->m_ops[i]->getOutputs()).c_str());
    }
    if(buf && capacity > out.size())
        memcpy(buf, out.c_str(), out.size() + 1);
    return (int)out.size();
}

// A host window that stays open over steps
void *probe_access(void *tensor_box) { return (*(std::shared_ptr<Tensor> *)tensor_box)->access().release(); }
void *probe_access_data(void *ta) { return ((TensorAccess *)ta)->data(); }
void probe_access_close(void *ta) { delete(TensorAccess *)ta; }
// the device buffer of a batched tensor that the operations of the last step read
void *probe_last_batch(void *tensor_box)
{
    auto *t = dynamic_cast<HipTensor *>(((std::shared_ptr<Tensor> *)tensor_box)->get());
    auto *db = static_cast<HipDoubleBuffer *>(t->m_storage.get());
    return db->m_dev[db->m_index ^ 1];
}

}  // extern "C"
