#!/usr/bin/env python3
"""Writes src/kernels.rs -- the safe `Kernels` dispatch layer of the local-hip crate -- from include/local_hip.h.

    python3 local-hip/gen_safe.py            # rewrites local-hip/src/kernels.rs
    python3 local-hip/gen_safe.py --check    # exit 1 when src/kernels.rs is not what the header generates

The reference binds its GPU layer method by method in local-metal/src/kernels.rs: `Kernels::<op>_into(&self,
&mut CommandBatch, &MetalBuffer.., u32 scalars) -> Result<()>` (e.g. kernels.rs:4819, 5176, 5434), plus blocking forms
that take the context.  Every LH_API function of the header whose first parameter is the batch or the context and
whose other parameters are buffers, buffer arrays and scalars is such an operation: it gets one method with the
header's name less the `lh_` prefix, the header's parameter names in the header's order (which the header documents
against the reference method by method), forwarding to `ffi::lh_<op>` and turning the status into `Error`.  No Rust
toolchain exists where this library is built, so the file is generated and checked textually
(tests/test_ffi_binding.py), never compiled there."""
from __future__ import annotations

import os
import re
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
import gen_ffi  # noqa: E402  (the header parser)

OUT = os.path.join(HERE, "src", "kernels.rs")
BY_HAND = os.path.join(HERE, "src", "lib.rs")

# C parameter type -> (Rust parameter type, expression passed to the raw function)
SCALAR = {"uint32_t": "u32", "uint64_t": "u64", "size_t": "usize", "float": "f32", "int": "c_int",
          "lh_quant": "ffi::lh_quant", "lh_dtype": "ffi::lh_dtype"}
NOT_OPS = ("lh_context_", "lh_buffer_", "lh_batch_", "lh_event_", "lh_graph_", "lh_debug_", "lh_last_error", "lh_version")


def squeeze(ctype: str) -> str:
    return " ".join(ctype.replace("*", " * ").split()).replace(" *", "*")


def wrap(name, ret, params):
    """Rust source of the method for one header function, or None when it is not a dispatch operation."""
    if name.startswith(NOT_OPS) or ret != "int" or not params:
        return None
    first_t, first_n = squeeze(params[0][0]), params[0][1]
    if first_t == "lh_batch*":
        head, first_arg = "batch: &mut CommandBatch", "batch.as_ptr()"
    elif first_t == "lh_context*":
        head, first_arg = "ctx: &Context", "ctx.as_ptr()"
    else:
        return None
    sig, pre, args = [head], [], [first_arg]
    for ctype, pname in params[1:]:
        t = squeeze(ctype)
        pn = pname + "_" if pname in gen_ffi.RUST_KEYWORDS else pname
        if t in ("const lh_buffer*", "lh_buffer*"):
            sig.append(f"{pn}: &Buffer")
            args.append(f"{pn}.as_ptr()")
        elif t in ("const lh_buffer* const*", "lh_buffer* const*"):
            sig.append(f"{pn}: &[&Buffer]")
            pre.append(f"        let {pn}_raw: Vec<*{'const' if t.startswith('const') else 'mut'} ffi::lh_buffer> = "
                       f"{pn}.iter().map(|b| b.as_ptr(){'' if not t.startswith('const') else ' as *const ffi::lh_buffer'}).collect();")
            args.append(f"{pn}_raw.as_ptr()")
        elif t == "const uint32_t*":
            sig.append(f"{pn}: &[u32]")
            args.append(f"{pn}.as_ptr()")
        elif t in SCALAR:
            sig.append(f"{pn}: {SCALAR[t]}")
            args.append(pn)
        else:
            return None      # host pointers and the like: not a dispatch operation
    method = name[len("lh_"):]
    body = [f"    /// `{name}` (include/local_hip.h)."]
    if len(sig) > 7:
        body.append("    #[allow(clippy::too_many_arguments)]")
    body.append(f"    pub fn {method}(&self, {', '.join(sig)}) -> Result<()> {{")
    body.extend(pre)
    body.append("        // SAFETY: every pointer comes from a live handle of this crate; the library validates sizes and shapes.")
    body.append(f"        check(unsafe {{ ffi::{name}({', '.join(args)}) }})")
    body.append("    }")
    return "\n".join(body)


def generate(text: str) -> str:
    fns = gen_ffi.parse_header(text)
    with open(BY_HAND) as f:
        by_hand = set(re.findall(r"ffi::(lh_\w+)\(", f.read()))
    methods, skipped = [], []
    for name, ret, params in fns:
        src = wrap(name, ret, params)
        if src:
            methods.append(src)
        elif not name.startswith(NOT_OPS):
            skipped.append(name)
            if params and squeeze(params[0][0]) in ("lh_batch*", "lh_context*") and name not in by_hand:
                raise SystemExit(f"{name} is a dispatch operation that the header's types alone do not wrap: it needs a wrapper in src/lib.rs")
    lines = [
        "// The kernel-dispatch layer: `Kernels`, one method per operation of liblocal_hip.so, with the names and the argument",
        "// order that local-engine calls on local-metal (local-metal/src/kernels.rs).  GENERATED by gen_safe.py from",
        "// include/local_hip.h: do not edit.  Operations with host pointers and the helpers of the codec are wrapped by hand in lib.rs: " +
        ", ".join(n for n in skipped if n in by_hand) + ".",
        "// Other host-side helpers are reached through `ffi`: " + ", ".join(n for n in skipped if n not in by_hand) + ".",
        "use core::ffi::c_int;",
        "",
        "use crate::batch::CommandBatch;",
        "use crate::buffer::Buffer;",
        "use crate::context::Context;",
        "use crate::error::{check, Result};",
        "use crate::ffi;",
        "",
        "/// Stand-in for `local_metal::Kernels` (kernels.rs:116-219 builds ~95 Metal pipelines there; the HIP kernels are",
        "/// linked into the library, so this type holds nothing and `new` cannot fail for a missing shader).",
        "#[derive(Debug, Default, Clone, Copy)]",
        "pub struct Kernels;",
        "",
        "impl Kernels {",
        "    /// `Kernels::new(ctx, library)` of the reference; the context only proves that a gfx950 device was opened.",
        "    pub fn new(_ctx: &Context) -> Result<Self> {",
        "        Ok(Kernels)",
        "    }",
        "",
    ]
    lines.append("\n\n".join(methods))
    lines.append("}")
    return "\n".join(lines) + "\n"


def main() -> int:
    text = open(gen_ffi.HEADER).read()
    rust = generate(text)
    if "--check" in sys.argv:
        have = open(OUT).read() if os.path.exists(OUT) else ""
        if have != rust:
            print("local-hip/src/kernels.rs is out of date: run python3 local-hip/gen_safe.py", file=sys.stderr)
            return 1
        return 0
    with open(OUT, "w") as f:
        f.write(rust)
    print(f"wrote {OUT}: {rust.count('pub fn ') - 1} methods")
    return 0


if __name__ == "__main__":
    sys.exit(main())
